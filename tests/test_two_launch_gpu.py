"""A short decode step in two launches (pv_last_kernel): partial-row counts up to and past the rule's line, every padded count
of query heads, ragged residuals, both position forms -- against the forms that a call's flags name -- and the ring row that
its workgroups make from the logits, bit for bit the sum of the probabilities that the call returns."""
import ctypes

import pytest
import torch

from hqekv_amd import synth

pytestmark = pytest.mark.gpu


def _cache(dev, B, Hkv, blocks, residual, shuffled, seed):
    from hqekv_amd.pack_unpack import uniform_group_quantize_pack_last_dim
    n = 32 * sum(blocks)
    q, K, V = synth.make_qkv(B, 1, Hkv, n + residual, 128, seed, dev)
    tokens = torch.randperm(n if shuffled else n // 32, generator=torch.Generator().manual_seed(n))
    tokens = tokens if shuffled else (tokens[:, None] * 32 + torch.arange(32)).reshape(-1)
    classes, at = {}, 0
    for bits, c in zip((16, 8, 4, 2, 1), blocks):
        classes[bits] = tokens[at:at + 32 * c].sort()[0]
        at += 32 * c
    return synth.build_cache(K, V, classes, residual, uniform_group_quantize_pack_last_dim)


def _form(plan, extra=None):
    """1: two launches, 0: more."""
    from hqekv_amd import _lib
    return _lib.load().hqekv_selftest_step_form(plan.k_segs, plan.n_k, plan.v_segs, plan.n_v, plan.out.data_ptr(), plan.B, plan.Hq, plan.Hkv, plan.D,
                                                plan.Tall, plan.flags, extra)


@pytest.mark.parametrize("blocks,residual,rows", [((0, 0, 0, 1, 0), 0, 1), ((1, 1, 1, 1, 1), 3, 6), ((4, 8, 33, 17, 8), 1, 13),
                                                  ((8, 16, 40, 40, 16), 64, 19), ((8, 16, 40, 48, 16), 65, 20), ((8, 16, 40, 48, 16), 129, 21)])
@pytest.mark.parametrize("B,n_rep,Hkv,shuffled", [(1, 4, 8, False), (3, 3, 2, True), (2, 5, 4, False), (1, 8, 1, True), (2, 1, 5, True), (1, 2, 8, False)])
def test_against_the_separate_launches(dev, blocks, residual, rows, B, n_rep, Hkv, shuffled):
    from hqekv_amd import _lib
    from hqekv_amd.attention import DecodePlan, decode_attention
    pkv = _cache(dev, B, Hkv, blocks, residual, shuffled, 11)
    q = torch.randn(B, n_rep * Hkv, 1, 128, generator=torch.Generator(device=dev).manual_seed(3), device=dev, dtype=torch.float16)
    n = 32 * sum(blocks) + residual
    plan = DecodePlan(q, pkv)
    assert _lib.load().hqekv_pv_workspace_bytes(plan.v_segs, plan.n_v, B, n_rep * Hkv, Hkv, 128) == rows * B * n_rep * Hkv * 512
    assert _form(plan) == (1 if rows <= 20 else 0)
    w, o = decode_attention(q, pkv, None, n, zero_init=False, flags=_lib.FUSE_SOFTMAX)
    w2, o2 = decode_attention(q, pkv, None, n, zero_init=False, flags=_lib.FUSE_SOFTMAX | _lib.SEPARATE_COMBINE)
    # (fp32 sums in another order before the same fp16 roundings: a score moves by one place, its probability by 2^-10 x |score|)
    torch.testing.assert_close(w.float(), w2.float(), rtol=1e-2, atol=1e-5)
    torch.testing.assert_close(o.float(), o2.float(), rtol=1e-3, atol=2e-3)
    again = decode_attention(q, pkv, None, n, zero_init=False, flags=_lib.FUSE_SOFTMAX)
    assert torch.equal(w, again[0]) and torch.equal(o, again[1])


@pytest.mark.parametrize("B", [1, 2, 8])
@pytest.mark.parametrize("blocks,residual", [((0, 0, 0, 8, 0), 1), ((1, 1, 1, 1, 1), 3), ((4, 8, 33, 17, 8), 30), ((8, 16, 40, 40, 16), 2), ((8, 16, 40, 48, 16), 2)])
def test_ring_row_is_the_sum_of_the_returned_probabilities(dev, B, blocks, residual):
    from hqekv_amd import _lib, attention
    lib, Hq, Hkv, D = _lib.load(), 32, 8, 128
    pkv = _cache(dev, B, Hkv, blocks, residual, False, 12)
    q = torch.randn(B, Hq, 1, D, generator=torch.Generator(device=dev).manual_seed(4), device=dev, dtype=torch.float16)
    plan, n = attention.DecodePlan(q, pkv), 32 * sum(blocks) + residual
    line = torch.full((n + 3,), float("nan"), dtype=torch.float16, device=dev)
    w, o = torch.empty(B, Hq, 1, n, dtype=torch.float16, device=dev), torch.empty(B, Hq, 1, D, dtype=torch.float16, device=dev)
    x = _lib.StepExtra(ring_line=line.data_ptr(), ring_order=attention.ring_order(n, w))
    assert _form(plan, ctypes.byref(x)) == 1
    rc = lib.hqekv_decode_step(plan.k_segs, plan.n_k, plan.v_segs, plan.n_v, ctypes.c_void_p(q.data_ptr()), None, 0, ctypes.c_void_p(w.data_ptr()),
                               ctypes.c_void_p(o.data_ptr()), B, Hq, Hkv, D, n, ctypes.c_void_p(plan.ws.data_ptr()), plan.ws.numel() * 4, _lib.FUSE_SOFTMAX,
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ctypes.byref(x))
    assert rc == 0
    assert torch.equal(line[:n], w.sum(0).sum(0).view(-1)) and bool(line[n:].isnan().all())
    w2, o2 = plan.run(q)
    assert torch.equal(w, w2) and torch.equal(o, o2)


def test_replays_count_their_own_arrivals(dev):
    """The counters of the last arrival belong to a call: replays with eager calls between them."""
    from hqekv_amd.attention import DecodePlan
    pkv = _cache(dev, 2, 8, (1, 4, 9, 9, 1), 7, False, 13)
    q = torch.randn(2, 32, 1, 128, device=dev, dtype=torch.float16)
    plan = DecodePlan(q, pkv)
    assert _form(plan) == 1
    want = [x.clone() for x in plan.run(q)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        got = plan.run(q)
    for _ in range(4):
        for x in got:
            x.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        assert all(torch.equal(a, b) for a, b in zip(plan.run(q), want))
