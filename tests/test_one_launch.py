"""A short decode step in one launch (csrc/decode_step.hip): which calls take it, and that it writes what two launches write, bit for
bit, also where its workgroups wait for nobody and do what others would have left them."""
import ctypes

import pytest
import torch

from hqekv_amd import synth

D = 128


def _dense(n, k, v, slab=0):
    from hqekv_amd import _lib
    return ((_lib.Seg * 1)(_lib.Seg(bits=16, layout=_lib.LAYOUT_TOKEN_MAJOR, n_tokens=n, data=k, slab_tokens=slab)),
            (_lib.Seg * 1)(_lib.Seg(bits=16, n_tokens=n, data=v, slab_tokens=slab)))


def _one(segs, n, q=1 << 40, w=1 << 41, o=1 << 42, B=1, Hkv=4, rep=4, flags=None, extra=None):
    from hqekv_amd import _lib
    vp = ctypes.c_void_p
    rc = _lib.load().hqekv_selftest_step_one(segs[0], len(segs[0]), segs[1], len(segs[1]), vp(q), vp(w), vp(o), B, rep * Hkv, Hkv, D, n,
                                             _lib.FUSE_SOFTMAX if flags is None else flags, None if extra is None else ctypes.byref(extra))
    assert rc >= 0, _lib.load().hqekv_last_error()
    return rc


def test_lines_of_the_rule():
    from hqekv_amd import _lib
    k, v = 1 << 43, 1 << 44
    assert [_one(_dense(n, k, v), n) for n in (1, 2560, 2561)] == [1, 1, 0]           # 20 and 21 p.V units of 128
    assert [_one(_dense(640, k, v), 640, rep=r) for r in (1, 4, 5, 8, 9)] == [1, 1, 1, 1, 0]
    assert _one(_dense(640, k, v), 640, flags=0) == 0 and _one(_dense(640, k, v), 640, flags=_lib.FUSE_SOFTMAX | _lib.TWO_LAUNCHES) == 0
    two_bit = lambda n: (_lib.Seg * 1)(_lib.Seg(bits=2, n_tokens=n, data=v, scale=v + (1 << 30), zero=v + (1 << 31), idx=1 << 45))
    for n, want in ((4096, 1), (4160, 0)):                                              # 64 and 65 q.K^T tiles of 64 tokens
        assert _one((_dense(n, k, v)[0], two_bit(n)), n) == want


def test_what_q_and_k_are_read_from_is_not_written():
    """A step's output, probabilities and epilogue stand beside q.K^T's reads: over them, two launches."""
    from hqekv_amd import _lib
    k, v, n, slab, Hkv, rep = 1 << 43, 1 << 44, 64, 96, 4, 4
    segs, q, w, o = _dense(n, k, v, slab), 1 << 40, 1 << 41, 1 << 42
    row, q_end, k_end = 2 * D, q + rep * Hkv * 2 * D, k + (Hkv - 1) * slab * 2 * D + n * 2 * D
    assert _one(segs, n, o=q) == 0 and _one(segs, n, o=q_end - row) == 0 and _one(segs, n, o=q_end) == 1 and _one(segs, n, o=q - rep * Hkv * row) == 1
    assert _one(segs, n, w=q) == 0 and _one(segs, n, w=q_end) == 1
    assert _one(segs, n, o=k_end) == 1 and _one(segs, n, o=k_end - row) == 0 and _one(segs, n, w=k) == 0 and _one(segs, n, w=k_end) == 1

    def append(k_dst):
        return _lib.StepExtra(append_rows=1, new_k=1 << 46, new_v=1 << 47, k_dst=k_dst, v_dst=1 << 48, k_dst_slab_tokens=slab, v_dst_slab_tokens=slab)
    assert _one(segs, n, extra=append(k + n * row)) == 1 and _one(segs, n, extra=append(k + (n - 1) * row)) == 0
    assert _one(segs, n, extra=append(k - row)) == 1 and _one(segs, n, extra=append(k)) == 0
    ring = lambda at: _lib.StepExtra(ring_line=at, ring_order=1)
    assert _one(segs, n, extra=ring(k_end)) == 1 and _one(segs, n, extra=ring(k_end - 2)) == 0
    # a ring row past what rides along has a launch of its own behind the reads
    assert _one(_dense(n, k, v, slab), n, B=9, Hkv=8, extra=ring(k)) == 1


def _cache(dev, B, Hkv, blocks, residual, shuffled, low_uniform, seed):
    from hqekv_amd.pack_unpack import uniform_group_quantize_pack_last_dim
    n = 32 * sum(blocks)
    _, K, V = synth.make_qkv(B, 1, Hkv, n + residual, D, seed, dev)
    tokens = torch.randperm(n if shuffled else n // 32, generator=torch.Generator().manual_seed(n))
    tokens = tokens if shuffled else (tokens[:, None] * 32 + torch.arange(32)).reshape(-1)
    classes, at = {}, 0
    for bits, c in zip((16, 8, 4, 2, 1), blocks):
        classes[bits] = tokens[at:at + 32 * c].sort()[0]
        at += 32 * c
    return synth.build_cache(K, V, classes, residual, uniform_group_quantize_pack_last_dim)


@pytest.mark.gpu
@pytest.mark.parametrize("blocks,residual", [((0, 0, 0, 1, 0), 0), ((0, 1, 0, 0, 0), 1), ((1, 1, 1, 1, 1), 3), ((4, 8, 33, 17, 8), 1), ((8, 16, 40, 40, 16), 64),
                                             ((0, 0, 0, 0, 9), 2), ((5, 0, 0, 0, 0), 0), ((0, 9, 0, 0, 0), 31)])
@pytest.mark.parametrize("B,n_rep,Hkv,shuffled,low_uniform", [(1, 4, 8, False, True), (3, 3, 2, True, True), (2, 5, 4, False, False), (1, 8, 1, True, False),
                                                              (2, 1, 5, True, True), (1, 2, 8, False, False), (8, 4, 8, False, True), (2, 7, 3, False, True)])
def test_the_bits_of_two_launches(dev, blocks, residual, B, n_rep, Hkv, shuffled, low_uniform):
    from hqekv_amd import _lib
    from hqekv_amd.attention import DecodePlan
    pkv = _cache(dev, B, Hkv, blocks, residual, shuffled, low_uniform, 17)
    q = torch.randn(B, n_rep * Hkv, 1, D, generator=torch.Generator(device=dev).manual_seed(3), device=dev, dtype=torch.float16)
    got = []
    for more in (_lib.TWO_LAUNCHES, 0, _lib.IMPATIENT):
        plan = DecodePlan(q, pkv, low_uniform=low_uniform)
        plan.flags |= more
        assert _one((plan.k_segs, plan.v_segs), plan.Tall, q.data_ptr(), plan.weights.data_ptr(), plan.out.data_ptr(), B, Hkv, n_rep, plan.flags) == \
            (more != _lib.TWO_LAUNCHES)
        for _ in range(2):   # the second on memory that holds the first's numbers
            plan.weights.fill_(7)
            plan.out.fill_(7)
            plan.run(q)
        got.append((plan.weights, plan.out))
    for w, o in got[1:]:
        assert torch.equal(w, got[0][0]) and torch.equal(o, got[0][1])


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,blocks,residual", [(1, 32, 8, (0, 0, 0, 8, 0), 1), (2, 32, 8, (1, 1, 1, 1, 1), 3), (1, 40, 8, (4, 8, 33, 17, 8), 30), (8, 32, 8, (0, 2, 2, 2, 0), 5),
                                                      (1, 3, 3, (0, 0, 0, 2, 0), 1)])
def test_a_whole_step(dev, B, Hq, Hkv, blocks, residual):
    """The ring row and the appended rows beside the attention."""
    from hqekv_amd import _lib, attention
    lib = _lib.load()
    pkv = _cache(dev, B, Hkv, blocks, residual, False, True, 18)
    g = torch.Generator(device=dev).manual_seed(4)
    q, k, v = (torch.randn(B, h, 1, D, generator=g, device=dev, dtype=torch.float16) for h in (Hq, Hkv, Hkv))
    plan, n = attention.DecodePlan(q, pkv), 32 * sum(blocks) + residual
    got = []
    for more in (_lib.TWO_LAUNCHES, 0, _lib.IMPATIENT):
        line = torch.full((n + 3,), float("nan"), dtype=torch.float16, device=dev)
        w, o = torch.empty(B, Hq, 1, n, dtype=torch.float16, device=dev), torch.empty(B, Hq, 1, D, dtype=torch.float16, device=dev)
        kd, vd = torch.zeros(B, Hkv, 2, D, dtype=torch.float16, device=dev), torch.zeros(B, Hkv, 2, D, dtype=torch.float16, device=dev)
        x = _lib.StepExtra(ring_line=line.data_ptr(), ring_order=attention.ring_order(n, w), append_rows=1, new_k=k.data_ptr(), new_v=v.data_ptr(),
                           k_dst=kd.data_ptr() + 2 * D, v_dst=vd.data_ptr() + 2 * D, k_dst_slab_tokens=2, v_dst_slab_tokens=2)
        flags = plan.flags | more
        assert _one((plan.k_segs, plan.v_segs), n, q.data_ptr(), w.data_ptr(), o.data_ptr(), B, Hkv, Hq // Hkv, flags, x) == (more != _lib.TWO_LAUNCHES)
        rc = lib.hqekv_decode_step(plan.k_segs, plan.n_k, plan.v_segs, plan.n_v, q.data_ptr(), None, 0, w.data_ptr(), o.data_ptr(), B, Hq, Hkv, D, n,
                                   plan.ws.data_ptr(), plan.ws.numel() * 4, flags, torch.cuda.current_stream().cuda_stream, ctypes.byref(x))
        assert rc == 0, lib.hqekv_last_error()
        assert torch.equal(line[:n], w.sum(0).sum(0).view(-1)) and bool(line[n:].isnan().all())
        assert torch.equal(kd[:, :, 1:], k) and torch.equal(vd[:, :, 1:], v) and not bool(kd[:, :, 0].any()) and not bool(vd[:, :, 0].any())
        got.append((w, o, line[:n]))
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(other, got[0]))


@pytest.mark.gpu
def test_two_streams_at_once(dev):
    """Steps of two caches on two streams, each with its own workspace, share the chip."""
    from hqekv_amd.attention import DecodePlan
    plans, want = [], []
    for seed in (1, 2):
        pkv = _cache(dev, 16, 8, (1, 4, 9, 9, 1), 7, False, True, seed)
        q = torch.randn(16, 32, 1, D, generator=torch.Generator(device=dev).manual_seed(seed), device=dev, dtype=torch.float16)
        plans.append((DecodePlan(q, pkv), q))
        want.append([x.clone() for x in plans[-1][0].run(q)])
    streams = [torch.cuda.Stream() for _ in plans]
    torch.cuda.synchronize()
    for _ in range(30):
        for (plan, q), s in zip(plans, streams):
            with torch.cuda.stream(s):
                plan.run(q)
    torch.cuda.synchronize()
    for (plan, _), (w, o) in zip(plans, want):
        assert torch.equal(plan.weights, w) and torch.equal(plan.out, o)


@pytest.mark.gpu
def test_a_workspace_without_room_for_the_records(dev):
    """What two launches need is enough, with the same bits; less is refused."""
    from hqekv_amd import _lib
    from hqekv_amd.attention import DecodePlan
    lib, pkv = _lib.load(), _cache(dev, 2, 4, (1, 1, 9, 8, 1), 3, False, True, 5)
    q = torch.randn(2, 16, 1, D, generator=torch.Generator(device=dev).manual_seed(3), device=dev, dtype=torch.float16)
    plan = DecodePlan(q, pkv)
    plan.run(q)
    want = plan.weights.clone(), plan.out.clone()
    need = lib.hqekv_decode_workspace_bytes(plan.k_segs, len(plan.k_segs), plan.v_segs, len(plan.v_segs), 2, 16, 4, D)
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    low, high = 0, need // 256
    while high - low > 1:
        size = 256 * ((low + high) // 2)
        plan.weights.fill_(7)
        plan.out.fill_(7)
        rc = lib.hqekv_decode_attn(plan.k_segs, len(plan.k_segs), plan.v_segs, len(plan.v_segs), q.data_ptr(), None, 0, plan.weights.data_ptr(),
                                   plan.out.data_ptr(), 2, 16, 4, D, plan.Tall, ws.data_ptr(), size, plan.flags, torch.cuda.current_stream().cuda_stream)
        if rc == 0:
            assert torch.equal(plan.weights, want[0]) and torch.equal(plan.out, want[1]), size
            high = size // 256
        else:
            assert rc == -3   # HQEKV_E_WORKSPACE
            low = size // 256
    assert 0 < 256 * high < need
