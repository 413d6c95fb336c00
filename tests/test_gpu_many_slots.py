"""More than eight experts per token: the combines and the adapters' slot sums take the slots eight at
a time. Slot counts around the multiples of eight, ids outside the layer, with and without LoRA, the
forward, the input and weight gradients and the adapters' gradients against the float64 oracle."""
import types

import numpy as np
import pytest
import torch

import oracle
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def k():
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from lazylora_amd.native import kernel
    return kernel()


@pytest.mark.parametrize("r", (0, 8, 24))
@pytest.mark.parametrize("topk", (7, 8, 9, 15, 16, 17, 24, 25))
def test_slots(k, topk, r):
    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] top-{topk} rank {r}", flush=True)
    rng = np.random.default_rng(topk)
    E, N, D, F = 26, 37, 288, 160
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h, g = (rng.standard_normal((N, D)).astype(np.float32) for _ in range(2))
    idx = np.stack([rng.permutation(E)[:topk] for _ in range(N)])
    idx[3, topk // 2], idx[5, topk - 1] = -1, E
    w = rng.uniform(0.2, 1.0, (N, topk)).astype(np.float32)
    lo = adapters = None
    if r:
        A = lambda n_in, n_out: (0.05 * rng.standard_normal((r, n_in)).astype(np.float32),
                                 0.05 * rng.standard_normal((n_out, r)).astype(np.float32))
        parts = A(D, F), A(D, F), A(F, D)
        lo = oracle.LoRA(*[v for p in parts for v in p])
        adapters = tuple(types.SimpleNamespace(lora_A=torch.from_numpy(a).cuda(), lora_B=torch.from_numpy(b).cuda(),
                                               scaling=2.0, dropout_rate=0.0) for a, b in parts)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    c = lambda a: torch.from_numpy(a).cuda()
    out = k.routed_forward(c(h), c(idx), c(w), L, lora=adapters)
    got = k.routed_backward(c(h), c(idx), c(w), L, c(g), lora=adapters)
    keep = (idx >= 0) & (idx < E)
    idx0, w0 = np.where(keep, idx, 0), np.where(keep, w, 0)
    # a skipped slot as expert 0 with weight 0 adds nothing to out, grad_h and the adapters
    assert_close(out.cpu().numpy(), oracle.routed_forward(h, idx0, w0, ex, lora=lo), "out")
    want = oracle.routed_backward(h, idx0, w0, ex, g, lora=lo)
    assert_close(got[0].cpu().numpy(), want[0], "grad_h")
    gw = got[1].cpu().numpy()
    assert (gw[~keep] == 0).all()
    assert_close(gw[keep], want[1][keep], "grad_w")
    for name, a, b in zip(("gate_A", "gate_B", "up_A", "up_B", "down_A", "down_B"), got[2] if r else (), want[2] if r else ()):
        assert_close(a.cpu().numpy(), b, name)
