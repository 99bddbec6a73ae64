"""The sum of p.V's partial rows (pv_rows_sum_kernel): chunk counts around what its threads hold, one and two workgroups per
row, on data whose sums are exact in any order."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv", [(1, 4, 1), (3, 32, 8), (1, 15, 3), (2, 32, 2)])
@pytest.mark.parametrize("chunks", [1, 2, 7, 8, 9, 31, 32, 33, 40, 41, 64, 65, 103, 257])
def test_exact_sums(dev, B, Hq, Hkv, chunks):
    """Probabilities of 2^-6 and zero, values of small integers: every partial sum is a multiple of 2^-6 below 2^13."""
    from hqekv_amd import _lib
    lib, D, n = _lib.load(), 128, 128 * chunks - 5   # 128 tokens to a chunk of fp16 rows; the last one ragged
    g = torch.Generator().manual_seed(chunks)
    v = torch.randint(-4, 5, (B, Hkv, n, D), generator=g).to(dev, torch.float16)
    p = (torch.randint(0, 2, (B, Hq, n), generator=g).to(dev, torch.float16) / 64).contiguous()
    s = _lib.Seg(bits=16, n_tokens=n, data=v.data_ptr(), scale=None, zero=None, idx=None, pos_base=0, layout=0, slab_tokens=0)
    segs = (_lib.Seg * 1)(s)
    ws = torch.empty(lib.hqekv_pv_workspace_bytes(segs, 1, B, Hq, Hkv, D), dtype=torch.uint8, device=dev)
    # (past what the chip holds at once -- six workgroups per CU, three above eight heads -- a workgroup takes several chunks)
    rows = ws.numel() // (B * Hq * 512)
    assert rows == chunks if B * Hkv * chunks <= (1536 if Hq // Hkv <= 8 else 768) else 1 < rows < chunks
    assert lib.hqekv_selftest_form(3, B * Hq, rows, 0) == (8 if B * Hq < 96 and rows > 40 else 32)
    out = torch.full((B, Hq, D), float("nan"), dtype=torch.float16, device=dev)
    rc = lib.hqekv_pv_hybrid(segs, 1, ctypes.c_void_p(p.data_ptr()), ctypes.c_void_p(out.data_ptr()), B, Hq, Hkv, D, n,
                             ctypes.c_void_p(ws.data_ptr()), ws.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    exact = (p.double().cpu().view(B, Hkv, Hq // Hkv, n, 1) * v.double().cpu().unsqueeze(2)).sum(3).view(B, Hq, D)
    assert torch.equal(out.cpu(), exact.half())
