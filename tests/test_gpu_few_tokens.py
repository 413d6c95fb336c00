"""The routed layer with so few (token, expert) pairs that its forward splits the contraction over
the waves of a work-group: pair counts on both sides of that line, one expert for all and many,
contraction lengths on and off 512, both layouts, activations with a third term, scale bytes that
zero their blocks, ids outside the layer, with and without LoRA, against the float64 oracle."""
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


@pytest.mark.parametrize("D,F", ((512, 512), (1024, 2560), (288, 96), (4608, 256)))
@pytest.mark.parametrize("N,topk", ((1, 1), (1, 8), (3, 2), (16, 1), (33, 1), (40, 4)))
@pytest.mark.parametrize("kind", ("normal", "forward layout", "outliers", "dead scales", "lora", "one expert"))
def test_few_pairs(k, D, F, N, topk, kind):
    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] N {N} top-{topk} D {D} F {F} {kind}", flush=True)
    rng = np.random.default_rng(N * topk + D + F)
    E = 9
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h = rng.standard_normal((N, D)).astype(np.float32)
    if kind == "outliers":
        h[:, 7::61] *= 1000.0
    if kind == "dead scales":
        for s in (ex.w1s, ex.w3s, ex.w2s):
            s[rng.random(s.shape) < 0.05] = 253 + int(rng.integers(0, 3))
    idx = np.stack([rng.permutation(E)[:topk] for _ in range(N)])
    if kind == "one expert":
        idx[:] = 4
    if kind == "normal" and N > 1:
        idx[0, 0] = E  # outside the layer: contributes nothing
    w = rng.uniform(0.5, 1.0, (N, topk)).astype(np.float32)
    lo = adapters = None
    if kind == "lora":
        A = lambda n_in, n_out: (0.05 * rng.standard_normal((4, n_in)).astype(np.float32),
                                 0.05 * rng.standard_normal((n_out, 4)).astype(np.float32))
        parts = A(D, F), A(D, F), A(F, D)
        lo = oracle.LoRA(*[v for p in parts for v in p])
        adapters = tuple(types.SimpleNamespace(lora_A=torch.from_numpy(a).cuda(), lora_B=torch.from_numpy(b).cuda(),
                                               scaling=2.0, dropout_rate=0.0) for a, b in parts)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    if kind == "forward layout":
        L.prepare_forward_layout()
    c = lambda a: torch.from_numpy(a).cuda()
    act = "situ" if N % 2 else "swiglu"
    got = k.routed_forward(c(h), c(idx), c(w), L, act=act, lora=adapters).cpu().numpy()
    keep = (idx >= 0) & (idx < E)
    want = oracle.routed_forward(h, np.where(keep, idx, 0), np.where(keep, w, 0), ex, act=act, lora=lo)
    assert_close(got, want, "out")


def test_line_from_the_checkpoint_layout(k):
    """Two tokens at top-8 of 7168 / 2048 experts are past the line: split-K items of the gate/up product
    would be four rounds of the chip. They take the one-tile items that a larger batch takes, and a row's
    result does not depend on the rows beside it there, so it is the batch's bit for bit (split-K adds
    the products of a row in another order)."""
    from lazylora_amd.experts import ExpertLayer
    E, D, F, N, topk = 16, 7168, 2048, 18, 8
    print(f"\n[case] 2 of {N} tokens, top-{topk} of {E}, D {D} F {F}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    mat = lambda R, K: (torch.randint(0, 256, (E, R, K // 2), dtype=torch.uint8, device="cuda", generator=gen),
                        torch.randint(117, 122, (E, R, K // 32), dtype=torch.uint8, device="cuda", generator=gen))
    L = ExpertLayer(*mat(F, D), *mat(F, D), *mat(D, F))
    h = torch.randn((N, D), device="cuda", generator=gen)
    w, idx = torch.topk(torch.rand((N, E), device="cuda", generator=gen), topk)
    w, idx = w.contiguous(), idx.contiguous()
    all_rows = k.routed_forward(h, idx, w, L)
    assert torch.equal(k.routed_forward(h[:2].contiguous(), idx[:2].contiguous(), w[:2].contiguous(), L), all_rows[:2])
