"""The strip kernel (csrc/kxw4_strip.hip) at the edges of its tiles, stages
and split plans, against the oracle: int32 partials and the order of every
FP32 step are fixed, so the outputs must be the oracle's bits."""
import ctypes as C

import numpy as np
import pytest
import torch

from knivesysl_xe_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(autouse=True, scope="module")
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    O.set_num_threads(16)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


# group, activation block, scale encoding
MODES = {"token128": (128, 0, O.SCALE_FP16), "token64": (64, 0, O.SCALE_FP16),
         "block32": (32, 32, O.SCALE_FP16_ZP4), "block64": (64, 32, O.SCALE_FP16_ZP4), "w8": (32, 32, None),
         "k16": (16, 32, O.SCALE_FP16_ZP4)}


def weight(rng, mode, M, K):
    group, _, enc = MODES[mode]
    lim = (-128, 128) if mode == "w8" else (-8, 8)
    codes = rng.integers(*lim, (M, K)).astype(np.int8)
    scales = (np.abs(rng.standard_normal((M, K // group))) * 0.02).astype(np.float16).view(np.uint16)
    if enc == O.SCALE_FP16_ZP4:
        scales = ((scales & 0xFFF0) | (rng.integers(-8, 8, scales.shape) & 0xF)).astype(np.uint16)
    bits = dev(scales.view(np.int16))
    w = ops.W4Weight.from_codes_s8(dev(codes), bits) if mode == "w8" else ops.W4Weight.from_codes(dev(codes), bits, group, enc)
    return codes, scales, w


def oracle(mode, codes, scales, act, variant, splits, **kw):
    group, block, enc = MODES[mode]
    return O.project(codes, scales, group, O.SCALE_S8 if mode == "w8" else enc, *act, block, variant, splits, **kw)


def check(y, ref, what):
    bits = np.uint16 if y.dtype == torch.bfloat16 else np.uint32
    got = (y.view(torch.int16) if y.dtype == torch.bfloat16 else y).cpu().numpy().view(bits)
    assert np.array_equal(got, ref.view(bits)), f"{what}: {np.count_nonzero(got != ref.view(bits))} of {got.size} differ"


def launches(call):
    """Kernel launches of `call`, counted as the nodes of its captured graph."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        call()
    n = C.c_size_t()
    assert C.CDLL(path).hipGraphGetNodes(C.c_void_p(g.raw_cuda_graph()), None, C.byref(n)) == 0
    return n.value


# tokens around the tile sizes (1, 2, 8, 16, 32); one K tile, an odd number of
# tiles (a half-empty last stage) and enough for whole stages; row-groups that
# do not divide the row waves; splits that end inside a tile (K = 640: 20 K32
# units in 16 parts) and splits with no unit at all (K = 128 in 16)
@pytest.mark.parametrize("mode", ["token128", "token64", "block32", "block64", "w8"])
@pytest.mark.parametrize("T,M,K,forced", [
    (1, 16, 128, 1), (2, 48, 384, 2), (3, 80, 640, 16), (8, 144, 640, 4), (9, 16, 128, 16), (16, 80, 1152, 8),
    (17, 48, 384, 1), (31, 80, 640, 2), (33, 144, 1152, 16), (64, 16, 640, 4), (70, 176, 384, 1), (130, 48, 640, 8)])
def test_strip_gemm_edges(mode, T, M, K, forced):
    rng = np.random.default_rng(T * M + K)
    codes, scales, w = weight(rng, mode, M, K)
    block = MODES[mode][1]
    x = rng.standard_normal((T, K)).astype(np.float32)
    res = rng.standard_normal((T, M)).astype(np.float32)
    a, act = ops.quantize_act(dev(x), block), O.quantize_act(x, block)
    sp = O.segment_splits(T, M, K, None, forced)
    check(ops.gemm(w, a, residual=dev(res), forced_splits=forced),
          oracle(mode, codes, scales, act, O.VAR_GEMM, sp, residual=res), f"{mode} T={T}")
    check(ops.gemm(w, a, torch.bfloat16, forced_splits=forced),
          oracle(mode, codes, scales, act, O.VAR_GEMM, sp, out_bf16=True), f"{mode} T={T} bf16")


# the GEMV's two accumulators, the K16 halves and the fan-out's association
@pytest.mark.parametrize("mode,T,M,K,splits", [
    ("token128", 1, 48, 640, 1), ("token128", 40, 80, 384, 2), ("token64", 2, 80, 1152, 8), ("token64", 33, 48, 640, 16),
    ("block32", 1, 80, 640, 16), ("block64", 17, 48, 384, 1), ("block32", 64, 16, 1152, 4), ("w8", 1, 48, 384, 2),
    ("w8", 16, 80, 640, 16), ("k16", 1, 48, 640, 16), ("k16", 2, 80, 384, 1), ("k16", 8, 16, 1152, 8),
    ("k16", 16, 144, 128, 4)])
def test_strip_gemv(mode, T, M, K, splits):
    rng = np.random.default_rng(T * M + K + splits)
    codes, scales, w = weight(rng, mode, M, K)
    block = MODES[mode][1]
    x = rng.standard_normal((T, K)).astype(np.float32)
    a, act = ops.quantize_act(dev(x), block), O.quantize_act(x, block)
    check(ops.gemv(w, a, splits=splits), oracle(mode, codes, scales, act, O.VAR_GEMV, splits), f"{mode} gemv")
    if mode not in ("w8", "k16"):
        c2, s2, w2 = weight(rng, mode, 32, K)
        ys = ops.gemv_fanout([w, w2], a)
        S = O.gemv_splits((M + 32) // 16)
        for c, s, y in ((codes, scales, ys[0]), (c2, s2, ys[1])):
            check(y, oracle(mode, c, s, act, O.VAR_FANOUT, S), f"{mode} fan-out")


# packed prompts whose segments have different split counts, and weights of a
# fan-out that are planned apart: strips of several split counts, over token
# ranges that start and end anywhere
@pytest.mark.parametrize("mode", ["token128", "token64", "block32", "w8"])
@pytest.mark.parametrize("rows,segs", [([4096], [9, 61, 300, 5]), ([8192, 48], [70, 3, 129]), ([1024, 2048], [250, 17, 40])])
def test_strip_packed_segments(mode, rows, segs):
    rng = np.random.default_rng(sum(rows) + sum(segs))
    K, T = 384, sum(segs)
    off = [0] + [int(o) for o in np.cumsum(segs)]
    block = MODES[mode][1]
    ws = [weight(rng, mode, M, K) for M in rows]
    x = rng.standard_normal((T, K)).astype(np.float32)
    a, act = ops.quantize_act(dev(x), block), O.quantize_act(x, block)
    ys = ops.gemm_fanout([w for _, _, w in ws], a, offsets=off)
    for (c, s, _), y in zip(ws, ys):
        sp = O.segment_splits(T, c.shape[0], K, off)
        check(y, oracle(mode, c, s, act, O.VAR_GEMM, sp), f"{mode} rows={c.shape[0]}")


# either side of the lines between the strip, the row-wave and the K-parallel
# kernel (csrc/kxw4_route.hpp): the first and last rows against the oracle,
# with the whole weight's split plan
@pytest.mark.parametrize("mode,call,T,M,K", [
    ("token64", "gemm", 5, 8192, 256), ("token64", "gemm", 5, 8176, 256), ("token128", "gemm", 4, 16400, 256),
    ("token128", "gemm", 4, 16384, 256), ("token128", "gemm", 3, 8192, 8192), ("token128", "gemm", 2, 16400, 256),
    ("token64", "gemm", 16, 8208, 12288),
    ("token64", "gemv", 4, 48, 8320), ("token64", "gemv", 5, 48, 8320), ("token128", "gemv", 1, 48, 8192),
    ("token128", "gemv", 2, 8192, 8320), ("token128", "gemv", 1, 8208, 8320),
    ("w8", "gemm", 8, 117984, 4608), ("w8", "gemm", 9, 117984, 4608), ("w8", "gemv", 1, 131072, 4608),
    # one and two splits of one or two tokens, four splits, sixteen splits on
    # either side of the K-parallel kernel's slices, K past its LDS, reference
    # mode with many rows, and full rounds of W8 rows
    ("token128", "gemm", 1, 32784, 2560), ("token128", "gemm", 2, 20496, 2432), ("token64", "gemm", 2, 8192, 4096),
    ("token64", "gemm", 2, 8208, 4096), ("token64", "gemm", 8, 14336, 6144), ("token64", "gemm", 12, 6144, 4608),
    ("token64", "gemm", 8, 592, 7936), ("token64", "gemm", 8, 640, 6144), ("token64", "gemm", 4, 3072, 17408),
    ("token128", "gemm", 4, 1024, 1152), ("token128", "gemm", 5, 1024, 2176), ("token128", "gemv", 4, 4096, 4224),
    ("token64", "gemm", 1, 48, 49280), ("token128", "gemm", 1, 48, 98432),
    ("block64", "gemm", 4, 32784, 640), ("block64", "gemm", 2, 32784, 640), ("block32", "gemm", 8, 24576, 4096),
    ("block64", "gemm", 8, 24592, 4096), ("block64", "gemv", 3, 65536, 384),
    ("w8", "gemm", 9, 57344, 4608), ("w8", "gemm", 8, 57344, 4608), ("w8", "gemm", 2, 245760, 4608)])
def test_strip_rowwave_line(mode, call, T, M, K):
    group, block, enc = MODES[mode]
    g = torch.Generator(device=DEV).manual_seed(T * M + K)
    lim = (-128, 128) if mode == "w8" else (-8, 8)
    codes = torch.randint(*lim, (M, K), generator=g, device=DEV, dtype=torch.int8)
    bits = (0.02 * torch.rand(M, K // group, generator=g, device=DEV)).to(torch.float16).view(torch.int16)
    w = ops.W4Weight.from_codes_s8(codes, bits) if mode == "w8" else ops.W4Weight.from_codes(codes, bits, group, enc)
    x = torch.randn(T, K, generator=g, device=DEV).cpu().numpy()
    a, act = ops.quantize_act(dev(x), block), O.quantize_act(x, block)
    if call == "gemm":
        y, var, sp = ops.gemm(w, a), O.VAR_GEMM, O.segment_splits(T, M, K)
    else:
        y, var, sp = ops.gemv(w, a), O.VAR_GEMV, O.gemv_splits(M // 16)
    for lo in (0, M - 48):
        c, s = codes[lo:lo + 48].cpu().numpy(), bits[lo:lo + 48].cpu().numpy().view(np.uint16)
        check(y[:, lo:lo + 48].contiguous(), oracle(mode, c, s, act, var, sp), f"{mode} {call} T={T} M={M} K={K} row {lo}")


# long K at 8 and 16 tokens: the row-wave kernel's LDS does not hold the
# activations, and one launch that reads the weight once takes all of them
@pytest.mark.parametrize("mode,T", [("w8", 8), ("w8", 16), ("k16", 8), ("k16", 16)])
def test_long_k_reads_the_weight_once(mode, T):
    rng = np.random.default_rng(900 + T)
    M, K = 80, 17408
    codes, scales, w = weight(rng, mode, M, K)
    x = rng.standard_normal((T, K)).astype(np.float32)
    a, act = ops.quantize_act(dev(x), 32), O.quantize_act(x, 32)
    want = oracle(mode, codes, scales, act, O.VAR_GEMV, O.gemv_splits(M // 16))
    for option in (0, 2):                                # the default dispatch, the row-wave kernel preferred
        with ops.option("decode_kernel", option):
            y = ops.gemv(w, a)
            check(y, want, f"{mode} T={T}")
            assert launches(lambda: ops.gemv(w, a, out=y)) == 1


# Packed prompts past the strip kernel's limit: split segments on the strips,
# each run of one-split segments on the large tiles as a projection of its own
# (t0 > 0, weights left out, residual and BF16 rows shifted with it), what is
# too small for the tiles in one strip launch, few-token entries apart from the
# others in a deep grid, split counts that fill 32-token tiles apart, and plans
# that the general kernel takes in one launch. `n` is the launches that shows
# which way a plan went; the first and last rows go against the oracle.
@pytest.mark.parametrize("mode,rows,K,segs,n", [
    ("token64", [8192], 384, [3, 700, 5, 600], 3), ("token128", [8192], 384, [3, 700, 5, 600], 3),
    ("block32", [8192], 384, [3, 700, 5, 600], 3), ("block64", [8192], 384, [9, 700, 5, 600], 3),
    ("token64", [1024, 32768], 1024, [200, 400, 230], 4), ("block32", [1024, 32768], 384, [200, 400, 230], 4),
    ("token128", [1024, 32768], 1024, [200, 400, 230], 4),
    ("block32", [3568, 3568], 384, [34, 1, 121, 250, 19, 14, 1], 3),
    ("token64", [5344, 5344], 1920, [123, 48, 119, 33, 6, 39], 1),
    ("token128", [9008, 9008], 4096, [100, 1, 100, 1, 100], 1),
    ("token128", [8192], 384, [20, 20, 20, 20, 3], 2), ("block32", [8192], 384, [20, 20, 20, 20, 3], 2),
    ("w8", [8192], 384, [20, 20, 20, 20, 3], 2)])
def test_packed_beside_the_large_tiles(mode, rows, K, segs, n):
    group, block, enc = MODES[mode]
    g = torch.Generator(device=DEV).manual_seed(sum(rows) + sum(segs))
    lim = (-128, 128) if mode == "w8" else (-8, 8)
    T, off = sum(segs), [0] + [int(o) for o in np.cumsum(segs)]
    ws = []
    for M in rows:
        codes = torch.randint(*lim, (M, K), generator=g, device=DEV, dtype=torch.int8)
        bits = (0.02 * torch.rand(M, K // group, generator=g, device=DEV)).to(torch.float16).view(torch.int16)
        w = ops.W4Weight.from_codes_s8(codes, bits) if mode == "w8" else ops.W4Weight.from_codes(codes, bits, group, enc)
        ws.append((codes, bits, w))
    x = torch.randn(T, K, generator=g, device=DEV).cpu().numpy()
    a, act = ops.quantize_act(dev(x), block), O.quantize_act(x, block)
    res = torch.randn(T, rows[0], generator=g, device=DEV)
    for out in (torch.float32, torch.bfloat16):
        if len(rows) == 1:
            y = ops.gemm(ws[0][2], a, out, residual=res, offsets=off)
            assert launches(lambda: ops.gemm(ws[0][2], a, out, residual=res, offsets=off, out=y)) == n
            ys = [y]
        else:
            ys = ops.gemm_fanout([w for _, _, w in ws], a, out, offsets=off)
            assert launches(lambda: ops.gemm_fanout([w for _, _, w in ws], a, out, offsets=off, outs=ys)) == n
        for (codes, bits, _), y in zip(ws, ys):
            M = codes.shape[0]
            sp = O.segment_splits(T, M, K, off)
            for lo in (0, M - 48):
                c, s = codes[lo:lo + 48].cpu().numpy(), bits[lo:lo + 48].cpu().numpy().view(np.uint16)
                kw = {"residual": res[:, lo:lo + 48].contiguous().cpu().numpy()} if len(rows) == 1 else {}
                check(y[:, lo:lo + 48].contiguous(),
                      oracle(mode, c, s, act, O.VAR_GEMM, sp, out_bf16=out == torch.bfloat16, **kw),
                      f"{mode} rows={M} from {lo} {out}")


# 32-token tiles of two and four splits, a partial last tile, with residual
@pytest.mark.parametrize("mode", ["token128", "token64", "block32", "block64", "w8"])
@pytest.mark.parametrize("forced", [2, 4])
def test_strip_split_32_token_tiles(mode, forced):
    M, K, T = 8192, 640, 70
    rng = np.random.default_rng(forced)
    codes, scales, w = weight(rng, mode, M, K)
    x = rng.standard_normal((T, K)).astype(np.float32)
    res = rng.standard_normal((T, M)).astype(np.float32)
    block = MODES[mode][1]
    a, act = ops.quantize_act(dev(x), block), O.quantize_act(x, block)
    sp = O.segment_splits(T, M, K, None, forced)
    y = ops.gemm(w, a, residual=dev(res), forced_splits=forced)
    for lo in (0, M - 48):
        check(y[:, lo:lo + 48].contiguous(),
              oracle(mode, codes[lo:lo + 48], scales[lo:lo + 48], act, O.VAR_GEMM, sp,
                     residual=np.ascontiguousarray(res[:, lo:lo + 48])), f"{mode} forced {forced} rows from {lo}")


# the modes that reach the other decode kernels by option only (decode_kernel:
# 1 K-parallel, 2 row-wave), and the general GEMM's W8 path
@pytest.mark.parametrize("kernel", [1, 2])
@pytest.mark.parametrize("mode", ["block32", "block64", "w8", "k16"])
@pytest.mark.parametrize("T,M,K,S", [(1, 80, 640, 16), (2, 48, 384, 1), (3, 144, 1152, 8), (8, 80, 640, 2), (9, 48, 384, 4),
                                     (16, 144, 640, 8)])
def test_other_decode_kernels(mode, kernel, T, M, K, S):
    rng = np.random.default_rng(T * M + K + S)
    codes, scales, w = weight(rng, mode, M, K)
    x = rng.standard_normal((T, K)).astype(np.float32)
    res = rng.standard_normal((T, M)).astype(np.float32)
    a, act = ops.quantize_act(dev(x), 32), O.quantize_act(x, 32)
    with ops.option("decode_kernel", kernel):
        check(ops.gemv(w, a, residual=dev(res), splits=S), oracle(mode, codes, scales, act, O.VAR_GEMV, S, residual=res),
              f"{mode} gemv")
        if mode == "k16":
            return
        sp = O.segment_splits(T, M, K, None, S)
        check(ops.gemm(w, a, torch.bfloat16, forced_splits=S),
              oracle(mode, codes, scales, act, O.VAR_GEMM, sp, out_bf16=True), f"{mode} gemm")
        if mode != "w8":
            ys = ops.gemv_fanout([w, w], a)
            ref = oracle(mode, codes, scales, act, O.VAR_FANOUT, O.gemv_splits(2 * M // 16))
            for y in ys:
                check(y, ref, f"{mode} fan-out")


@pytest.mark.parametrize("T,M,K,forced", [(65, 144, 640, 1), (70, 80, 384, 4), (200, 2064, 256, 0)])
def test_w8_general_gemm(T, M, K, forced):
    rng = np.random.default_rng(T + M)
    codes, scales, w = weight(rng, "w8", M, K)
    x = rng.standard_normal((T, K)).astype(np.float32)
    res = rng.standard_normal((T, M)).astype(np.float32)
    a, act = ops.quantize_act(dev(x), 32), O.quantize_act(x, 32)
    sp = O.segment_splits(T, M, K, None, forced)
    with ops.option("gemm_kernel", 1):
        check(ops.gemm(w, a, residual=dev(res), forced_splits=forced),
              oracle("w8", codes, scales, act, O.VAR_GEMM, sp, residual=res), f"T={T}")
