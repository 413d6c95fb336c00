"""The routed backward at the edges of its transposed products' epilogues: row counts around the
staged halves and pairs of a 16-row tile and around the large-bucket groups (49 rows and more),
feature and hidden widths that end inside a 256- or 128-column stripe, both activations, with and
without the LoRA term of the W2 epilogue, against the float64 oracle at the path's bar."""
import types

import numpy as np
import pytest
import torch

import oracle
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu

ROWS = (1, 7, 8, 9, 15, 16, 17, 49, 63, 64, 81)  # tokens of expert 0, 1, ...


@pytest.fixture(scope="module")
def k():
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from lazylora_amd.native import kernel
    return kernel()


@pytest.mark.parametrize("layouts", (False, True))
@pytest.mark.parametrize("D,F", ((256, 32), (288, 256), (512, 384), (256, 544), (1024, 1024)))
@pytest.mark.parametrize("act,r", (("swiglu", 0), ("situ", 0), ("situ", 8)))
def test_epilogue_edges(k, D, F, act, r, layouts):
    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] D {D} F {F} {act} rank {r} layouts {layouts}", flush=True)
    rng = np.random.default_rng(D + F)
    E, N = len(ROWS), sum(ROWS)
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h = rng.standard_normal((N, D)).astype(np.float32)
    idx = np.repeat(np.arange(E), ROWS)[rng.permutation(N)].reshape(N, 1)
    w = rng.uniform(0.5, 1.0, (N, 1)).astype(np.float32)
    g = rng.standard_normal((N, D)).astype(np.float32)
    lo = None
    adapters = None
    if r:
        A = lambda n_in, n_out: (0.05 * rng.standard_normal((r, n_in)).astype(np.float32),
                                 0.05 * rng.standard_normal((n_out, r)).astype(np.float32), 2.0)
        parts = A(D, F), A(D, F), A(F, D)
        lo = oracle.LoRA(*[v for p in parts for v in p[:2]])
        adapters = tuple(types.SimpleNamespace(lora_A=torch.from_numpy(a).cuda(), lora_B=torch.from_numpy(b).cuda(),
                                               scaling=s, dropout_rate=0.0) for a, b, s in parts)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    if layouts:
        L.prepare_forward_layout()
        L.prepare_backward_layout()
    c = lambda a: torch.from_numpy(a).cuda()
    got = k.routed_backward(c(h), c(idx), c(w), L, c(g), act=act, lora=adapters)
    want = oracle.routed_backward(h, idx, w, ex, g, act=act, lora=lo) if lo else oracle.routed_backward(h, idx, w, ex, g, act=act)
    assert_close(got[0].cpu().numpy(), want[0], "grad_h")
    assert_close(got[1].cpu().numpy(), want[1], "grad_w")
    for e, n in enumerate(ROWS):  # no bucket hides in the others
        rows = idx[:, 0] == e
        assert_close(got[0].cpu().numpy()[rows], want[0][rows], f"grad_h of the expert with {n} rows")
