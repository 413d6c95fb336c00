"""The quantisers read x in 32-byte (fp32) and 16-byte (bf16) pieces, and x need only be 8- and 4-byte
aligned: the routed forward at the C entry with x at such addresses, at widths around a super-chunk,
with outlier channels (third terms), token rows and bucket tiles alike, bit for bit the result from
an aligned x. The single-matrix products likewise: x at every 8 bytes, and the transposed product's
gradient, which it reads in 32-byte pieces or splits in a pass of its own, at every 4."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def k():
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from lazylora_amd.native import kernel
    return kernel()


@pytest.mark.parametrize("bf16", (False, True))
@pytest.mark.parametrize("E,N,topk", ((5, 9, 3), (2, 150, 1)))  # short buckets; large ones only
@pytest.mark.parametrize("D", (32, 480, 512, 544, 1024))
def test_offsets(k, D, E, N, topk, bf16):
    from lazylora_amd.experts import ExpertLayer
    from lazylora_amd.native import BF16, F32, I64
    print(f"\n[case] D {D} {E} experts, {N} tokens, top-{topk}, bf16 {bf16}", flush=True)
    rng = np.random.default_rng(D + N)
    ex = oracle.random_experts(rng, E, D, 96, 117, 121)
    L = ExpertLayer(*[torch.from_numpy(a).cuda() for a in (ex.w1p, ex.w1s, ex.w3p, ex.w3s, ex.w2p, ex.w2s)])
    x = rng.standard_normal((N, D)).astype(np.float32)
    x[:, 7::97] *= 1000.0
    h = torch.from_numpy(x).cuda().to(torch.bfloat16 if bf16 else torch.float32)
    idx = torch.from_numpy(np.stack([rng.permutation(E)[:topk] for _ in range(N)])).cuda()
    w = torch.from_numpy(rng.uniform(0.5, 1.0, (N, topk)).astype(np.float32)).cuda()
    nws = int(k.lib.mxfp4_moe_workspace_size(N, topk, E, D, 96))
    outs = []
    for off in (0, 2, 4, 6):  # elements: 8 bytes of fp32, 4 of bf16, at a time
        buf = torch.zeros(N * D + 16, dtype=h.dtype, device="cuda")
        buf[off:off + N * D] = h.reshape(-1)
        ws = torch.empty(nws, dtype=torch.uint8, device="cuda")
        out = torch.empty((N, D), dtype=torch.float32, device="cuda")
        rc = k.lib.mxfp4_moe_forward_fl(
            out.data_ptr(), buf.data_ptr() + off * buf.element_size(), BF16 if bf16 else F32, idx.data_ptr(), I64,
            w.data_ptr(), N, topk, *L.pointers(), None, E, D, 96, 0, None, None, 0, 0, ws.data_ptr(), nws,
            torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        outs.append(out)
    for off, out in zip((2, 4, 6), outs[1:]):
        assert torch.equal(out, outs[0]), off


@pytest.mark.parametrize("M", (1, 17, 256, 257))  # both sides of the products' few-row kernels
@pytest.mark.parametrize("R,K", ((512, 96), (500, 512), (96, 1056)))
def test_product_offsets(k, R, K, M):
    print(f"\n[case] M {M} R {R} K {K}", flush=True)
    rng = np.random.default_rng(M + R + K)
    packed, scales = (torch.from_numpy(a).cuda() for a in (rng.integers(0, 256, (R, K // 2), dtype=np.uint8),
                                                           rng.integers(117, 122, (R, K // 32), dtype=np.uint8)))
    stream = torch.cuda.current_stream().cuda_stream
    for name, n_in, n_out, step in (("gemm", K, R, 2), ("gemm_t", R, K, 1)):
        x = torch.from_numpy(rng.standard_normal((M, n_in)).astype(np.float32)).cuda()
        nws = int(getattr(k.lib, f"mxfp4_{name}_workspace_size")(M, K, R))
        outs = []
        for off in range(0, 8, step):  # elements of 4 bytes
            buf = torch.zeros(M * n_in + 16, dtype=torch.float32, device="cuda")
            buf[off:off + M * n_in] = x.reshape(-1)
            ws = torch.empty(nws, dtype=torch.uint8, device="cuda")
            y = torch.zeros((M, n_out), dtype=torch.float32, device="cuda")
            rc = getattr(k.lib, f"mxfp4_{name}")(y.data_ptr(), buf.data_ptr() + 4 * off, packed.data_ptr(),
                                                 scales.data_ptr(), M, K, R, ws.data_ptr(), nws, stream)
            assert rc == 0
            outs.append(y)
        assert torch.isfinite(outs[0]).all() and outs[0].abs().max() > 0
        for off, y in zip(range(step, 8, step), outs[1:]):
            assert torch.equal(y, outs[0]), (name, off)
