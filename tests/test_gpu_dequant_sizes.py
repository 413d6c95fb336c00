"""Dequantisation at sizes around the pieces a work-group writes (one block, a few, past one and past
several work-groups), fp32 and bf16, every scale byte, and from and to pointers that only the
block-wise kernel takes (codes at an odd byte, output at 4 bytes), bit for bit against the oracle."""
import ctypes

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


@pytest.mark.parametrize("offset", (0, 1))
@pytest.mark.parametrize("bf16", (False, True))
@pytest.mark.parametrize("R,K", ((1, 32), (3, 32), (7, 224), (64, 128), (33, 1056), (257, 96), (1, 8192)))
def test_sizes(k, R, K, bf16, offset):
    print(f"\n[case] dequant [{R}, {K}] bf16 {bf16} offset {offset}", flush=True)
    rng = np.random.default_rng(R + K)
    p, s = oracle.random_mx(rng, (R, K), 0, 255)
    buf = torch.zeros(p.size + 16, dtype=torch.uint8, device="cuda")
    buf[offset:offset + p.size] = torch.from_numpy(p).cuda().reshape(-1)
    S = torch.from_numpy(s).cuda()
    words = R * K // 2 if bf16 else R * K  # 32-bit words of the output, one guard word on either side
    out = torch.full((words + 8,), 0x5A5A5A5A, dtype=torch.int32, device="cuda")
    fn = k.lib.mxfp4_dequant_bf16 if bf16 else k.lib.mxfp4_dequant
    at = 4 + (1 if offset else 0)
    rc = fn(ctypes.c_void_p(out.data_ptr() + 4 * at), ctypes.c_void_p(buf.data_ptr() + offset),
            ctypes.c_void_p(S.data_ptr()), K, R, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    got = out.cpu().numpy()
    want = oracle.dequant(p, s)
    want = (torch.from_numpy(want).to(torch.bfloat16).view(torch.int16).numpy() if bf16 else want).reshape(-1).view(np.int32)
    assert np.array_equal(got[at:at + words], want)
    assert (got[:at] == 0x5A5A5A5A).all() and (got[at + words:] == 0x5A5A5A5A).all()
