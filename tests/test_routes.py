"""The dispatch rule of the decode launches (csrc/kxw4_route.hpp), on the CPU:
each shape goes to the kernel that was measured ahead on it (launches of a
graph replay with the weights from HBM on an MI355X; strip / other kernel in
us beside the case)."""
import ctypes as C
import os
import subprocess

import pytest

from oracle import oracle as O

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "knivesysl_xe_amd", "csrc")
STRIP, ROWWAVE, KPARALLEL = 0, 1, 2
CUS = 256


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    src, out = d / "route.cpp", d / "route.so"
    src.write_text('#include "kxw4_route.hpp"\n'
                   'extern "C" int route(int rgs, int T, int K, int group, int S, int blocks, int w8) {\n'
                   f'    return kxw4::decode_route({{{CUS}, rgs, T, K, group, S, blocks != 0, w8 != 0}});\n'
                   '}\n'
                   'extern "C" int packed(int K, int group, int launches, int tile_runs, long long few, long long lots,\n'
                   '                      long long strips, long long tile_work, long long general) {\n'
                   f'    return kxw4::packed_general({{{CUS}, K, group, launches, tile_runs, few, lots, strips, tile_work,'
                   ' general});\n'
                   '}\n'
                   'extern "C" int wide(long long rows, int T) {\n'
                   f'    return kxw4::gemmr_wide({CUS}, rows, T);\n'
                   '}\n'
                   'extern "C" int small_tile(long long rows, int T) {\n'
                   f'    return kxw4::w4a4_small({CUS}, rows, T);\n'
                   '}\n'
                   'extern "C" long long limit(int block, int group) { return kxw4::one_split_strips(block, group); }\n')
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", str(out)],
                   check=True)
    lib = C.CDLL(str(out))
    lib.packed.argtypes = [C.c_int] * 4 + [C.c_longlong] * 5
    lib.limit.restype = C.c_longlong
    lib.wide.argtypes = lib.small_tile.argtypes = [C.c_longlong, C.c_int]
    return lib


@pytest.fixture(scope="module")
def route(rules):
    return rules.route


def splits(call, M, K, T):
    return O.gemv_splits(M // 16) if call != "gemm" else int(O.gemm_splits(M // 16, (T + 7) // 8, K // 32, 0))


@pytest.mark.parametrize("group,call,M,K,T,want", [
    # one or two splits
    (128, "gemm", 32768, 5120, 1, ROWWAVE),              # 19.8 / 16.2
    (128, "gemm", 32768, 5120, 2, ROWWAVE),              # 20.4 / 16.4
    (128, "gemm", 17408, 5120, 1, ROWWAVE),              # 12.2 / 10.9
    (128, "gemm", 17408, 5120, 2, ROWWAVE),              # 14.0 / 11.1
    (64, "gemm", 16384, 2048, 2, ROWWAVE),               # 8.1 / 6.9
    (64, "gemm", 34816, 5120, 16, ROWWAVE),              # 24.2 / 20.4
    (64, "gemv", 65536, 5120, 2, ROWWAVE),               # 36.5 / 33.3
    (128, "gemm", 28480, 2432, 1, STRIP),                # 9.7 / 10.8
    # four splits
    (128, "gemm", 10240, 12288, 1, ROWWAVE),             # 14.5 / 13.5
    (128, "gemm", 10240, 12288, 2, ROWWAVE),             # 15.5 / 13.8
    (64, "gemm", 8192, 5120, 1, ROWWAVE),                # 8.1 / 7.4
    (64, "gemm", 14336, 8192, 8, ROWWAVE),               # 17.4 / 15.3
    (128, "gemm", 6144, 2048, 4, STRIP),                 # 5.8 / 7.6
    # many rows in eight splits: a GEMV or a fan-out, not the GEMM's lines
    (64, "gemv", 24576, 5120, 4, STRIP),                 # 21.1 / 25.7
    (128, "gemv", 34816, 5120, 8, STRIP),                # 30.0 / 37.3
    (64, "gemv", 17408, 5120, 1, STRIP),                 # 12.9 / 18.2
    # one or two row-groups per CU, long rows
    (64, "gemm", 6144, 12288, 8, ROWWAVE),               # 14.2 / 12.7
    (64, "gemv", 6144, 12288, 12, ROWWAVE),              # 15.6 / 13.3
    (64, "gemv", 2048, 8192, 1, ROWWAVE),                # 6.8 / 5.6
    (128, "gemv", 2048, 12288, 4, KPARALLEL),            # 8.7 / 8.0
    (128, "gemv", 4096, 4096, 4, STRIP),
    (64, "gemv", 4096, 4096, 2, ROWWAVE),                # 5.8 / 5.6
    # few rows in sixteen splits
    (128, "gemm", 1024, 12288, 1, KPARALLEL),            # 8.3 / 6.8
    (64, "gemm", 592, 7936, 8, KPARALLEL),               # 9.0 / 7.5: two slices of four tokens
    (64, "gemm", 640, 6144, 8, STRIP),                   # 7.7 / 9.2: one slice of eight
    (64, "gemm", 3072, 17408, 4, STRIP),                 # 12.4 / 15.9: more slices than CUs
])
def test_per_token(route, group, call, M, K, T, want):
    assert route(M // 16, T, K, group, splits(call, M, K, T), 0, 0) == want


@pytest.mark.parametrize("group,call,M,K,T,want", [
    (64, "gemm", 34816, 5120, 4, ROWWAVE),               # 32.4 / 29.8
    (64, "gemm", 24576, 8192, 4, ROWWAVE),               # 31.9 / 28.6
    (32, "gemm", 24576, 8192, 4, ROWWAVE),               # 32.4 / 30.3
    (32, "gemm", 34816, 5120, 4, STRIP),
    (64, "gemm", 26624, 8192, 8, STRIP),
    (64, "gemm", 34816, 5120, 1, STRIP),                 # 26.5 / 30.5
    (32, "gemv", 17408, 5120, 1, STRIP),                 # 15.2 / 30.2
])
def test_blocks(route, group, call, M, K, T, want):
    assert route(M // 16, T, K, group, splits(call, M, K, T), 1, 0) == want


@pytest.mark.parametrize("M,K,T,want", [
    (248320, 5120, 8, ROWWAVE),                          # 239 / 233
    (245760, 5120, 1, ROWWAVE),
    (393216, 5120, 12, ROWWAVE),                         # 393 / 379
    (65536, 5120, 12, ROWWAVE),                          # 76 / 71
    (57344, 8192, 16, ROWWAVE),
    (122880, 8192, 4, ROWWAVE),                          # 196 / 187
    (65536, 5120, 8, STRIP),
    (131072, 5120, 8, STRIP),                            # tie
    (200000, 5120, 1, STRIP),                            # 189 / 210
    (294912, 5120, 8, STRIP),                            # 291 / 292
    (248320, 4096, 1, STRIP),
])
def test_w8(route, M, K, T, want):
    assert route(M // 16, T, K, 32, splits("gemm", M, K, T), 1, 1) == want


def test_other_plans_stay_on_the_strips(route):
    assert route(2176, 17, 5120, 128, 1, 0, 0) == STRIP      # more than 16 tokens
    assert route(2176, 8, 5120, 128, 0, 0, 0) == STRIP       # split counts that differ
    assert route(320, 1, 17408, 16, 8, 1, 0) == STRIP        # K16


# (rows of each weight, K, segments; us on the strips and tiles / on the general kernel)
@pytest.mark.parametrize("group,rows,K,segs,want", [
    (64, [5344, 5344], 1920, [123, 48, 119, 33, 6, 39], True),           # 54.8 / 37.3
    (128, [9008, 9008], 4096, [100, 1, 100, 1, 100], True),              # 100 / 75
    (128, [17408], 5120, [100, 1, 100, 1, 100], True),                   # 120 / 95
    (64, [7952, 7952], 12160, [132, 7, 6, 34], True),                    # 189 / 136
    (128, [1968], 8192, [154, 5], False),                                # 25 / 64
    (64, [5120], 5120, [16, 32, 64, 128, 256], False),                   # 45 / 64
    (64, [5120, 5120], 17408, [16, 32, 64, 128, 256], False),            # 234 / 296
    (128, [9008, 9008], 4096, [16, 32, 64, 128, 256], False),            # 64 / 113
    (64, [9968], 4352, [14, 239, 239], False),                           # 62 / 88
])
def test_packed_prompts(rules, group, rows, K, segs, want):
    rgs, limit = [M // 16 for M in rows], rules.limit(0, group)
    S = [int(O.gemm_splits(rgs[0], (t + 7) // 8, K // 32, 0)) for t in segs]
    runs, open_ = [], False
    for t, s in zip(segs, S):
        if s == 1:
            runs = runs[:-1] + [runs[-1] + t] if open_ else runs + [t]
        open_ = s == 1
    strips = lambda t: sum(rgs) * -(-t // 32)
    tiles = [t for t in runs if strips(t) > limit] if sum(map(strips, runs)) > limit else []
    rest = sum(strips(t) for t in runs if t not in tiles)
    few = sum(sum(rgs) for t, s in zip(segs, S) if s > 1 and t <= 8)
    lots = sum(sum(rgs) * -(-t // 16) for t, s in zip(segs, S) if s > 1 and t > 8)
    launches = len(tiles) + (rest > 0) + (few > 0) + (lots > 0)
    general = sum(-(-r // 8) for r in rgs) * -(-sum(segs) // 64)
    assert bool(rules.packed(K, group, launches, len(tiles), few, lots, rest, sum(rgs) * sum(tiles), general)) == want


# one split: strips or large tiles (us on strips / on tiles)
@pytest.mark.parametrize("block,group,M,T,strips", [
    (0, 64, 17408, 96, False),                           # K = 5120: 33.1 / 29.8
    (0, 64, 14336, 128, False),                          # K = 4096: 27.0 / 24.9
    (0, 64, 10000, 192, False),                          # K = 1152: 13.2 / 11.4
    (0, 64, 5120, 256, True),                            # K = 17408
    (0, 128, 5120, 384, True),
    (0, 128, 17408, 128, False),                         # K = 5120: 35 / 35
    (32, 32, 5120, 512, True),                           # K = 17408: 227 / 234
    (32, 64, 17408, 256, False),                         # K = 5120: 113 / 109
])
def test_one_split_strips(rules, block, group, M, T, strips):
    assert (M // 16 * -(-T // 32) <= rules.limit(block, group)) == strips


# 64-token tiles or 32-token ones of the reference-mode GEMM, by the ratio of
# their times (64 / 32) measured at K = 5120
@pytest.mark.parametrize("M,T,wide", [
    (34816, 90, False),                                  # 1.20
    (17408, 210, False),                                 # 1.21
    (6544, 600, False),                                  # 1.17
    (8192, 384, False),                                  # 1.09
    (10240, 300, True),                                  # 0.92
    (17408, 300, True),                                  # 0.85
    (17408, 512, True),                                  # 0.92-0.96
    (12288, 700, True),                                  # 0.93
])
def test_reference_mode_tiles(rules, M, T, wide):
    assert bool(rules.wide((M // 16 + 7) // 8, T)) == wide


# 64 x 64 or 128 x 64 tiles of the W4A4 GEMM (us 64 x 64 / 128 x 64)
@pytest.mark.parametrize("M,T,small", [
    (5120, 64, True),                                    # K = 17408: 98 / 134
    (5120, 512, True),                                   # 154.7 / 179.8
    (5120, 2048, False),                                 # 463 / 441
    (2048, 1024, True),                                  # K = 5120: 40.2 / 42.7
    (8320, 84, True),                                    # K = 1408: 13.0 / 14.3
    (4096, 1024, False),                                 # two large for four small: 1.07
])
def test_w4a4_tiles(rules, M, T, small):
    assert bool(rules.small_tile((M // 16 + 3) // 4, T)) == small
