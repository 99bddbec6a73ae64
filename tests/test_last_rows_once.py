"""The probabilities of a prompt's last rows in one launch (slices of at most 128 keys): the same bits as in two, whether the
slices' statistics come from the other workgroups or a workgroup waits for nobody; each replay of a captured call equals the
call.  And the shorter prompts' launch at its edges of twelve waves."""
import ctypes as C

import pytest
import torch

from hqekv_amd import _lib


def _run(lib, q, k, R, patience, mask=None, size=1.0, ws=None):
    B, Hq, T, D = q.shape
    need = lib.hqekv_prompt_last_rows_workspace_bytes(B, Hq, T)
    ws = torch.full((need,), 0xff, dtype=torch.uint8, device=q.device) if ws is None else ws
    probs = torch.full((B, Hq, R, T), float("nan"), dtype=torch.float16, device=q.device)
    st = lambda t: (C.c_int64 * 3)(*t.stride()[:3])
    rc = lib.hqekv_selftest_last_rows(q.data_ptr(), st(q), k.data_ptr(), st(k), None if mask is None else mask.data_ptr(),
                                      None if mask is None else (C.c_int64 * 2)(mask.stride(0), mask.stride(2)), probs.data_ptr(), B, Hq, k.shape[1], T, D, R,
                                      128 ** -0.5, ws.data_ptr(), int(need * size), patience, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.hqekv_last_error()
    return probs


def test_workspace_holds_the_records_where_a_slice_is_a_tile_per_wave():
    need = _lib.load().hqekv_prompt_last_rows_workspace_bytes
    assert need(1, 32, 512) == 0
    assert need(1, 32, 513) == 32 * 5 * 32 * 16
    assert need(1, 32, 6144) == 32 * 48 * 32 * 16
    assert need(1, 32, 6145) == 32 * 48 * 32 * 8
    assert need(1, 16, 8192) == 16 * 64 * 32 * 8
    assert need(4, 32, 1536) == 128 * 12 * 32 * 16
    assert need(4, 32, 1537) == 128 * 12 * 32 * 8


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,T,R,masked", [
    (1, 32, 8, 513, 20, False),      # a key past four tiles; slices of four tiles, the last of one
    (1, 32, 8, 1003, 20, False),
    (1, 32, 8, 1024, 20, False),     # eight slices
    (1, 32, 8, 1025, 20, False),     # nine, the last of one key
    (1, 32, 8, 2048, 20, False),     # sixteen
    (1, 32, 8, 2049, 20, False),     # seventeen
    (1, 64, 4, 3072, 20, False),     # 24
    (1, 8, 2, 3073, 20, False),      # 25
    (1, 4, 1, 6144, 32, False),      # 48, the most
    (1, 32, 8, 4352, 20, False),     # 34: 27 744 pairs of workgroup and slice
    (1, 32, 8, 4609, 20, False),     # 37: 32 856, two launches
    (2, 28, 4, 545, 32, False),      # seven heads, all rows
    (1, 2, 2, 641, 1, False),        # one column
    (3, 40, 8, 640, 20, True),
    (16, 32, 8, 384 + 130, 20, True),   # three slices would be five: two launches
    (4, 32, 8, 1536, 20, True),
])
def test_one_launch_has_the_bits_of_two(B, Hq, Hkv, T, R, masked):
    lib, g = _lib.load(), torch.Generator("cuda").manual_seed(T)
    q, k = (torch.randn(B, H, T, 128, generator=g, device="cuda").half() for H in (Hq, Hkv))
    mask = None
    if masked:
        mask = torch.zeros(B, 1, R, T, device="cuda")
        mask[..., T // 2:] = -65504.0
        mask[0, :, R - 1] = float("-inf")   # (the floor makes this row even)
        mask = mask.half()
    two = _run(lib, q, k, R, -1, mask)
    assert torch.isfinite(two).all()
    # (half the size: room for the two launches' statistics, where the call is not two launches anyhow)
    for patience, size in ((2000, 1.0), (0, 1.0)) + (() if B == 16 else ((2000, 0.5),)):
        assert torch.equal(_run(lib, q, k, R, patience, mask, size).view(torch.int16), two.view(torch.int16)), (patience, size)
    # the workspace of a call before, whole of records with another launch's number
    ws = torch.zeros(lib.hqekv_prompt_last_rows_workspace_bytes(B, Hq, T), dtype=torch.uint8, device="cuda")
    _run(lib, q + 1, k, R, 2000, mask, ws=ws)
    assert torch.equal(_run(lib, q, k, R, 2000, mask, ws=ws).view(torch.int16), two.view(torch.int16))


@pytest.mark.gpu
def test_captured_call_is_replayed_on_new_inputs():
    lib, g = _lib.load(), torch.Generator("cuda").manual_seed(5)
    q, k = (torch.randn(1, H, 1003, 128, generator=g, device="cuda").half() for H in (32, 8))
    ws = torch.zeros(lib.hqekv_prompt_last_rows_workspace_bytes(1, 32, 1003), dtype=torch.uint8, device="cuda")
    _run(lib, q, k, 20, 2000, ws=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        probs = _run(lib, q, k, 20, 2000, ws=ws)
    for i in range(4):
        q.copy_(torch.randn(q.shape, generator=g, device="cuda"))
        graph.replay()
        assert torch.equal(probs.view(torch.int16), _run(lib, q, k, 20, 2000).view(torch.int16)), i


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,R", [(1, 32, 8, 20), (2, 7, 1, 32)])
@pytest.mark.parametrize("T", [257, 288, 353, 384, 385])
def test_twelve_waves(T, B, Hq, Hkv, R):
    """Tolerance: two roundings of a logit may fall to the other half -- the product's, 2^-5 below 64 and times the scale 2.8e-3, and
    the scaled one's, 2^-8 below 8 -- and the probability's own, 2^-11: 7.2e-3."""
    from hqekv_amd.prompt_attention import prompt_last_rows
    g = torch.Generator("cuda").manual_seed(T)
    q, k = (torch.randn(B, H, T, 128, generator=g, device="cuda").half() for H in (Hq, Hkv))
    got = prompt_last_rows(q, k, 128 ** -0.5, R)
    s = torch.matmul(q[:, :, T - R:].float(), k.float().repeat_interleave(Hq // Hkv, 1).transpose(2, 3).contiguous()).half()
    s = (s.float() * 128 ** -0.5).half().float().masked_fill(torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1)[T - R:], float("-inf"))
    torch.testing.assert_close(got.float(), s.softmax(-1), rtol=7.2e-3, atol=1e-6)
