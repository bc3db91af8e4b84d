"""The E2M3 repack kernels (csrc/kxw4_pack.hip) against the oracle, bit for
bit: every tier, one K tile and an odd number of tiles, block scales per 32
and per 128 columns, scales outside the range of the refined quotients
(subnormal, huge, zero, negative), groups of zeros, and a payload that does
not start on 16 bytes."""
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


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def both(tier, payload, bs, cols, M, K):
    if tier == "w8":
        want = O.repack_e2m3_s8(payload.cpu().numpy(), bs, cols, M, K)
        w = ops.W4Weight.repack_e2m3_s8(payload, dev(bs), cols, M, K)
    else:
        want = O.repack_e2m3(payload.cpu().numpy(), bs, cols, M, K, tier)
        w = ops.W4Weight.repack_e2m3(payload, dev(bs), cols, M, K, tier)
    codes, scales = w.unpack()
    assert np.array_equal(scales.cpu().numpy().view(np.uint16), want[1])
    assert np.array_equal(codes.cpu().numpy(), want[0])


@pytest.mark.parametrize("tier", [0, 1, 2, "w8"])
@pytest.mark.parametrize("M,K,per", [(16, 128, 128), (48, 384, 32), (144, 640, 128)])
@pytest.mark.parametrize("kind", ["plain", "wide", "zeros", "unaligned"])
def test_repack_edges(tier, M, K, per, kind):
    rng = np.random.default_rng(M + K)
    n = M * K * 3 // 4
    payload = rng.integers(0, 256, n, dtype=np.uint8)
    if kind == "zeros":
        payload[: n // 2] = 0
    bs = rng.uniform(0.001, 0.05, ((M + 127) // 128, K // per)).astype(np.float32)
    if kind == "wide":
        bs = (bs * np.float32(2.0) ** rng.integers(-140, 120, bs.shape)).astype(np.float32)
        bs.flat[0] = 0.0
        bs.flat[-1] = -0.01
    if kind == "unaligned":
        t = torch.empty(n + 3, dtype=torch.uint8, device=DEV)[3:]
        t.copy_(dev(payload))
    else:
        t = dev(payload)
    both(tier, t, bs.reshape(-1), K // per, M, K)
