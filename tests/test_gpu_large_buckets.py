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


@pytest.mark.parametrize("pairs_over_line", (0, -3))
@pytest.mark.parametrize("D,F", ((1024, 1056), (1056, 1024), (1536, 1024)))
@pytest.mark.parametrize("rank", (0, 8))
def test_no_one_tile_items(k, D, F, rank, pairs_over_line):
    """Top-3, on both sides of the 12 rows per expert from which the routing's counts decide whether a
    forward's buckets take wide items (short ones, as here, do not), and where only one of the two products
    has them (the other's K is no multiple of 512)."""
    import types

    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] D {D} F {F} rank {rank} pairs over the line {pairs_over_line}", flush=True)
    rng = np.random.default_rng(D + F + rank)
    E, topk = 7, 3
    N = (12 * E + pairs_over_line) // topk
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h, g = (rng.standard_normal((N, D)).astype(np.float32) for _ in range(2))
    idx = np.stack([np.array([0, 1 + t % 2, 3]) for t in range(N)])  # two buckets of N rows, two of N / 2
    idx[0], idx[1, 1] = [4, 5, 1], 5                                  # one row, two rows; expert 6 has none
    w = rng.uniform(0.2, 1.0, (N, topk)).astype(np.float32)
    lo = adapters = None
    if rank:
        A = lambda n_in, n_out: (0.05 * rng.standard_normal((rank, n_in)).astype(np.float32),
                                 0.05 * rng.standard_normal((n_out, rank)).astype(np.float32))
        parts = A(D, F), A(D, F), A(F, D)
        lo = oracle.LoRA(*[v for p in parts for v in p])
        adapters = tuple(types.SimpleNamespace(lora_A=torch.from_numpy(a).cuda(), lora_B=torch.from_numpy(b).cuda(),
                                               scaling=2.0, dropout_rate=0.0) for a, b in parts)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    c = lambda a: torch.from_numpy(a).cuda()
    out = k.routed_forward(c(h), c(idx), c(w), L, lora=adapters)
    got = k.routed_backward(c(h), c(idx), c(w), L, c(g), lora=adapters)
    assert_close(out.cpu().numpy(), oracle.routed_forward(h, idx, w, ex, lora=lo), "out")
    want = oracle.routed_backward(h, idx, w, ex, g, lora=lo)
    for name, a, b in zip(("grad_h", "grad_w"), got, want):
        assert_close(a.cpu().numpy(), b, name)


SHORT = (16, 17, 1, 20, 32, 15, 48, 16, 0, 33, 8, 16, 30, 2, 16, 5)


# (rows of expert 0, 1, .., wide groups from the checkpoint layout, from the forward layout)
@pytest.mark.parametrize("rows,none,forward", (
    (SHORT, 0, 0),                   # no bucket of four tiles, few tiles past the first: one-tile items
    (SHORT[:-1] + (49,), 15, 7),     # one large bucket: all that have rows, and those of two tiles and more
    ((17,) * 65 + (12,) * 10, 0, 0),   # 65 tiles past the first: below both lines
    ((17,) * 66 + (12,) * 10, 0, 66),  # past the forward layout's
    ((17,) * 80 + (12,) * 10, 0, 80),  # 80: at the checkpoint layout's
    ((17,) * 81 + (12,) * 10, 91, 81),  # past it
    ((22,) * 80, 80, 80),            # averages that settle it from the checkpoint layout
    (tuple(8 + n % 90 for n in range(90)), 90, 81),  # 52 rows on average: large whatever the counts
))
@pytest.mark.parametrize("forward_layout,rank", ((False, 8), (True, 0)))
def test_short_buckets(k, rows, none, forward, forward_layout, rank):
    """Which buckets take wide items (meta word 4, at the start of the workspace, counts their groups), and
    the results, on both sides of each line of that rule; buckets of one row among those that do."""
    import types

    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] {len(rows)} experts, {sum(rows)} rows, forward layout {forward_layout}, rank {rank}", flush=True)
    E, N, D, F = len(rows), sum(rows), 1024, 1024
    rng = np.random.default_rng(N)
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h, g = (rng.standard_normal((N, D)).astype(np.float32) for _ in range(2))
    idx = np.repeat(np.arange(E), rows)[rng.permutation(N)].reshape(N, 1)
    w = rng.uniform(0.5, 1.0, (N, 1)).astype(np.float32)
    lo = adapters = None
    if rank:
        A = lambda n_in, n_out: (0.05 * rng.standard_normal((rank, n_in)).astype(np.float32),
                                 0.05 * rng.standard_normal((n_out, rank)).astype(np.float32))
        parts = A(D, F), A(D, F), A(F, D)
        lo = oracle.LoRA(*[v for p in parts for v in p])
        adapters = tuple(types.SimpleNamespace(lora_A=torch.from_numpy(a).cuda(), lora_B=torch.from_numpy(b).cuda(),
                                               scaling=2.0, dropout_rate=0.0) for a, b in parts)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    if forward_layout:
        L.prepare_forward_layout()
    c = lambda a: torch.from_numpy(a).cuda()
    ws = torch.empty(k.moe_workspace_bytes(N, 1, E, D, F), dtype=torch.uint8, device="cuda")
    out = k.routed_forward(c(h), c(idx), c(w), L, lora=adapters, save_for_backward=True, workspace=ws)
    assert int(ws[:64].view(torch.int32)[4]) == (forward if forward_layout else none)
    want = oracle.routed_forward(h, idx, w, ex, lora=lo)
    got = out.cpu().numpy()
    for e in range(E):  # no bucket hides in the others
        if rows[e]:
            assert_close(got[idx[:, 0] == e], want[idx[:, 0] == e], f"expert with {rows[e]} rows")
    got = k.routed_backward(c(h), c(idx), c(w), L, c(g), lora=adapters, reuse_forward=True, workspace=ws)
    want = oracle.routed_backward(h, idx, w, ex, g, lora=lo)
    for name, a, b in zip(("grad_h", "grad_w"), got, want):
        assert_close(a.cpu().numpy(), b, name)


# (rows of expert 0, 1, .., groups of the transposed products' large buckets)
@pytest.mark.parametrize("rows,groups", (
    (SHORT, 0),                      # two experts of three tiles, none of four
    (SHORT[:-1] + (49,), 3),         # one of four: three groups
    ((33, 40, 48) * 22, 0),          # 66 of three tiles
    ((33, 40, 48) * 22 + (35,), 67),  # 67
    (tuple(8 + n % 90 for n in range(90)), 98),  # over 48 rows on average
))
@pytest.mark.parametrize("layout", (False, True))
def test_three_tile_groups(k, rows, groups, layout):
    """Which buckets of three tiles the transposed products give their large-bucket items (meta word 3, at the
    start of the workspace, counts the groups), and the gradients, on both sides of each line of that rule."""
    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] {len(rows)} experts, {sum(rows)} rows, backward layout {layout}", flush=True)
    E, N, D, F = len(rows), sum(rows), 1024, 1024
    rng = np.random.default_rng(N)
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h, g = (rng.standard_normal((N, D)).astype(np.float32) for _ in range(2))
    idx = np.repeat(np.arange(E), rows)[rng.permutation(N)].reshape(N, 1)
    w = rng.uniform(0.5, 1.0, (N, 1)).astype(np.float32)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    if layout:
        L.prepare_backward_layout()
    c = lambda a: torch.from_numpy(a).cuda()
    ws = torch.empty(k.moe_workspace_bytes(N, 1, E, D, F), dtype=torch.uint8, device="cuda")
    gh, gw = k.routed_backward(c(h), c(idx), c(w), L, c(g), workspace=ws)
    assert int(ws[:64].view(torch.int32)[3]) == groups
    gh, gw = gh.cpu().numpy(), gw.cpu().numpy()
    want = oracle.routed_backward(h, idx, w, ex, g)
    for e in range(E):
        if rows[e]:
            assert_close(gh[idx[:, 0] == e], want[0][idx[:, 0] == e], f"grad_h of the expert with {rows[e]} rows")
    assert_close(gw, want[1], "grad_w")


# tokens of expert 0, 1, ..: items of 12 column blocks in a grid of 256 work-groups
@pytest.mark.parametrize("rows", (
    (128, 129, 144, 128, 140, 130, 127, 113),  # 12 groups, 4 of one tile: 7 full ones cut in two
    (256, 16, 33),                             # two full groups, one and three tiles: cut in four
    (300,) * 8,                                # 24 groups, 288 items: a whole round, then partial groups only
    (128,) * 9 + (17,),                        # full groups and one of two tiles, cut in two
))
@pytest.mark.parametrize("forward_layout", (False, True))
def test_last_round_runs(k, rows, forward_layout):
    """The last round of the wide items cut into runs of tiles where work-groups for all of these would idle:
    the runs of the partial groups (meta words 12 and 13, at the start of the workspace) are no more than
    their tiles."""
    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] {rows} forward layout {forward_layout}", flush=True)
    E, N, D, F = len(rows), sum(rows), 512, 3072
    rng = np.random.default_rng(N)
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h = rng.standard_normal((N, D)).astype(np.float32)
    idx = np.repeat(np.arange(E), rows)[rng.permutation(N)].reshape(N, 1)
    w = rng.uniform(0.5, 1.0, (N, 1)).astype(np.float32)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    if forward_layout:
        L.prepare_forward_layout()
    c = lambda a: torch.from_numpy(a).cuda()
    ws = torch.empty(k.moe_workspace_bytes(N, 1, E, D, F), dtype=torch.uint8, device="cuda")
    got = k.routed_forward(c(h), c(idx), c(w), L, workspace=ws).cpu().numpy()
    tiles = [-(-n // 16) for n in rows]
    wide = [t for t in tiles if t >= (2 if forward_layout else 1)]
    meta = ws[:64].view(torch.int32).tolist()
    assert meta[4:6] == [sum(-(-t // 8) for t in wide), sum(t // 8 for t in wide)]
    assert meta[12:14] == [sum(min(t % 8, n) for t in wide) for n in (2, 4)]
    want = oracle.routed_forward(h, idx, w, ex)
    for e, n in enumerate(rows):
        assert_close(got[idx[:, 0] == e], want[idx[:, 0] == e], f"expert with {n} rows")


@pytest.mark.parametrize("topk", (2, 4, 5, 8))
@pytest.mark.parametrize("D", (512, 1056))
@pytest.mark.parametrize("bf16", (False, True))
def test_only_large_buckets(k, topk, D, bf16):
    """Every bucket large and every token in several tiles: up to four slots its tiles are quantised one by
    one and its row in the token-major layout is not written, from five on they are copied from it (at a width
    that the large-bucket items do not take there are no tiles). Outlier channels, whose blocks have a third
    term."""
    from lazylora_amd.experts import ExpertLayer
    print(f"\n[case] top-{topk} D {D} bf16 {bf16}", flush=True)
    E, N, F = 8, 300, 64
    rng = np.random.default_rng(topk + D)
    ex = oracle.random_experts(rng, E, D, F, 117, 121)
    h = rng.standard_normal((N, D)).astype(np.float32)
    h[:, 5::97] *= 1000.0
    H = torch.from_numpy(h).cuda().to(torch.bfloat16 if bf16 else torch.float32)
    idx = np.stack([(np.arange(topk) + t) % E for t in range(N)])
    w = rng.uniform(0.5, 1.0, (N, topk)).astype(np.float32)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    ws = torch.empty(k.moe_workspace_bytes(N, topk, E, D, F), dtype=torch.uint8, device="cuda").random_(0, 256)
    got = k.routed_forward(H, torch.from_numpy(idx).cuda(), torch.from_numpy(w).cuda(), L, workspace=ws)
    assert ws[:64].view(torch.int32)[2] == 0  # no bucket is small
    assert_close(got.cpu().numpy(), oracle.routed_forward(H.float().cpu().numpy(), idx, w, ex), "out")
