"""The products with few rows, which split the contraction over the waves of a work-group, at the
edges of their tiles: 1 to 256 rows around the 16-row tiles and the two-tile items, output widths
around the column blocks, contraction lengths of one super-chunk and less, on and off its multiples,
with and without scale bytes that zero their blocks; against the C restatement of the reference at
the path's bar, the transposed product at 1e-5 of it (its own precision is 3e-6)."""
import numpy as np
import pytest
import torch

import oracle
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu

ROWS = (1, 2, 15, 16, 17, 31, 33, 64, 100, 255, 256, 257)
SHAPES = ((1, 32), (16, 64), (17, 512), (100, 544), (260, 1056), (2048, 512), (1000, 1536), (3001, 224), (96, 7168))


@pytest.fixture(scope="module")
def k():
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from lazylora_amd.native import kernel
    return kernel()


def weights(rng, R, K, dead):
    p, s = oracle.random_mx(rng, (R, K), 117, 121)
    if dead:
        s[rng.random(s.shape) < 0.05] = 253 + int(rng.integers(0, 3))
    return p, s


@pytest.mark.parametrize("dead", (False, True))
@pytest.mark.parametrize("R,K", SHAPES)
def test_gemm(k, clib, R, K, dead):
    rng = np.random.default_rng(R + K)
    p, s = weights(rng, R, K, dead)
    P, S = torch.from_numpy(p).cuda(), torch.from_numpy(s).cuda()
    for M in ROWS:
        print(f"\n[case] gemm M {M} R {R} K {K} dead {dead}", flush=True)
        x = rng.standard_normal((M, K)).astype(np.float32)
        got = k.gemm(torch.from_numpy(x).cuda(), P, S)
        assert torch.equal(got, k.gemm(torch.from_numpy(x).cuda(), P, S))  # one order of the sums
        assert_close(got.cpu().numpy(), clib.gemm(x, p, s), f"M {M}")


@pytest.mark.parametrize("dead", (False, True))
@pytest.mark.parametrize("R,K", SHAPES)
def test_gemm_t(k, clib, R, K, dead):
    rng = np.random.default_rng(R + K)
    p, s = weights(rng, R, K, dead)
    P, S = torch.from_numpy(p).cuda(), torch.from_numpy(s).cuda()
    for M in ROWS:
        print(f"\n[case] gemm_t M {M} R {R} K {K} dead {dead}", flush=True)
        dy = rng.standard_normal((M, R)).astype(np.float32)
        got = k.gemm_t(torch.from_numpy(dy).cuda(), P, S)
        assert torch.equal(got, k.gemm_t(torch.from_numpy(dy).cuda(), P, S))
        assert_close(got.cpu().numpy(), clib.gemm_t(dy, p, s), f"M {M}", rel=1e-5, cos=0.99999)
