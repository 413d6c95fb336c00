"""Buckets around the tile counts at which the routed forward changes its work-groups (one-tile
items, wide groups of up to eight 16-row tiles, partial second groups), from the checkpoint and
from the forward layout, at widths where a work item's last column tiles are missing, with scale
bytes that zero their blocks and with activations that carry a third term, against the float64
oracle at the path's bar, bucket by bucket."""
import numpy as np
import pytest
import torch

import oracle
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu

ROWS = (1, 16, 17, 32, 33, 48, 49, 64, 65, 127, 128, 129, 144, 145, 200)  # tokens of expert 0, 1, ...


@pytest.fixture(scope="module")
def k():
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from lazylora_amd.native import kernel
    return kernel()


@pytest.mark.parametrize("forward_layout", (False, True))
@pytest.mark.parametrize("D,F", ((512, 512), (512, 544), (1024, 96), (1536, 1024), (2560, 160)))
@pytest.mark.parametrize("inputs", ("normal", "outliers", "dead scales"))
def test_bucket_sizes(k, D, F, inputs, forward_layout):
    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] D {D} F {F} {inputs} forward layout {forward_layout}", flush=True)
    rng = np.random.default_rng(D + F)
    E, N = len(ROWS), sum(ROWS)
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h = rng.standard_normal((N, D)).astype(np.float32)
    if inputs == "outliers":
        h[:, 5::97] *= 1000.0
    if inputs == "dead scales":
        for s in (ex.w1s, ex.w3s, ex.w2s):
            s[rng.random(s.shape) < 0.02] = 253 + int(rng.integers(0, 3))
    idx = np.repeat(np.arange(E), ROWS)[rng.permutation(N)].reshape(N, 1)
    w = rng.uniform(0.5, 1.0, (N, 1)).astype(np.float32)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    if forward_layout:
        L.prepare_forward_layout()
    c = lambda a: torch.from_numpy(a).cuda()
    got = k.routed_forward(c(h), c(idx), c(w), L).cpu().numpy()
    want = oracle.routed_forward(h, idx, w, ex)
    for e, n in enumerate(ROWS):  # no bucket hides in the others
        rows = idx[:, 0] == e
        assert_close(got[rows], want[rows], f"expert with {n} rows")
