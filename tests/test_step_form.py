"""Which launches a decode step takes (``hqekv_selftest_step_form``): what a step writes beside its attention rides in a short
step's p.V launch unless that launch reads the place it goes to -- then it gets a launch of its own, behind the reads."""
import ctypes
import random

import pytest
import torch

D = 128


def _rows(at, n, slab, slabs, row):
    """Addresses of the 16-byte pieces of n rows in each of `slabs` slabs."""
    return {at + s * slab * row + i for s in range(slabs) for i in range(0, n * row, 16)}


def _form(v, slabs, extra=None, out=1 << 40):
    """A step over ``v`` = [(address, tokens, slab, bits, idx address)], K covering as many positions elsewhere."""
    from hqekv_amd import _lib
    n = sum(e[1] for e in v)
    vs = (_lib.Seg * len(v))(*(_lib.Seg(bits=b, n_tokens=t, data=at, scale=None if b == 16 else at + (1 << 20), zero=None if b == 16 else at + (1 << 21),
                                        idx=idx, slab_tokens=slab) for at, t, slab, b, idx in v))
    ks = (_lib.Seg * 1)(_lib.Seg(bits=16, layout=_lib.LAYOUT_TOKEN_MAJOR, n_tokens=n, data=1 << 42))
    rc = _lib.load().hqekv_selftest_step_form(ks, 1, vs, len(v), ctypes.c_void_p(out), 1, 4 * slabs, slabs, D, n, _lib.FUSE_SOFTMAX,
                                              None if extra is None else ctypes.byref(extra))
    assert rc >= 0, _lib.load().hqekv_last_error()
    return rc


def _append(k_dst, v_dst, slab_k, slab_v, rows=1, **more):
    from hqekv_amd import _lib
    return _lib.StepExtra(append_rows=rows, new_k=1 << 43, new_v=1 << 44, k_dst=k_dst, v_dst=v_dst, k_dst_slab_tokens=slab_k, v_dst_slab_tokens=slab_v, **more)


def test_appends_over_rows_that_the_step_reads():
    """Rows at random places in and around a V segment, against sets of addresses."""
    rng, seen, base = random.Random(1), {1: 0, 2: 0}, 1 << 30
    for _ in range(4000):
        slabs, slab, rows = rng.randint(1, 4), rng.randint(1, 9), rng.randint(1, 3)
        n = rng.randint(1, slab)
        dst_slab = slab if rng.random() < .7 else max(rows, rng.randint(1, 9))
        if dst_slab < rows:
            continue
        dst = base + 16 * rng.randint(-16 * slab * slabs - 20, 16 * slab * slabs + 20)
        hit = bool(_rows(base, n, slab, slabs, 256) & _rows(dst, rows, dst_slab, slabs, 256))
        k_side = rng.random() < .3
        form = _form([(base, n, slab, 16, None)], slabs, _append(dst if k_side else 1 << 45, 1 << 45 if k_side else dst, dst_slab if k_side else 64,
                                                                 64 if k_side else dst_slab, rows))
        seen[form] += 1
        assert form == 2 if hit else form == 1 or (dst_slab != slab and slabs > 1)
    assert min(seen.values()) > 500


@pytest.mark.parametrize("bits", [8, 4, 2, 1])
def test_what_a_class_is_read_from(bits):
    """Codes, scales, zero points and positions of a class, the row that leaves a tail, the ring's row, the output."""
    from hqekv_amd import _lib
    base, slabs, slab, n, idx = 1 << 30, 2, 96, 64, 1 << 35
    v = [(base, n, slab, bits, idx)]
    row, params = 16 * bits, 8
    places = [(base, row), (base + (1 << 20), params), (base + (1 << 21), params)]
    for at, r in places:
        last = at + slab * r + n * r   # one past the last slab's rows
        assert _form(v, slabs, _lib.StepExtra(ring_line=last, ring_order=1)) == 1
        assert _form(v, slabs, _lib.StepExtra(ring_line=last - 2, ring_order=1)) == 2
    assert _form(v, slabs, _lib.StepExtra(ring_line=idx + 8 * n - 2, ring_order=1)) == 2
    assert _form(v, slabs, _lib.StepExtra(ring_line=idx + 8 * n, ring_order=1)) == 1
    for t in (n - 1, n):
        leave = dict(leave_bits=bits, leave_src=1 << 46, leave_slab_tokens=4, leave_code=base + t * row, leave_scale=base + (1 << 20) + t * params,
                     leave_zero=base + (1 << 21) + t * params, leave_dst_slab_tokens=slab)
        assert _form(v, slabs, _lib.StepExtra(**leave)) == (1 if t == n else 2)
        assert _form(v, slabs, _append(1 << 45, 1 << 47, 64, 64, **leave)) == (1 if t == n else 2)
    assert _form(v, slabs) == 1 and _form(v, slabs, out=base + slab * row) == 0 and _form(v, slabs, out=base + (slab + n) * row) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hkv,n", [(1, 8, 64), (2, 2, 63), (3, 8, 1000)])
def test_sliding_window_replaces_its_oldest_row(dev, B, Hkv, n):
    """The step's value goes where the window's oldest was, which this step still reads: bit for bit what a step does that
    puts it elsewhere, and replays of it."""
    from hqekv_amd import _lib
    lib, Hq = _lib.load(), 4 * Hkv
    g = torch.Generator(device=dev).manual_seed(n)
    q, k, v = (torch.randn(B, h, 1, D, generator=g, device=dev, dtype=torch.float16) for h in (Hq, Hkv, Hkv))
    kw, vw = (torch.randn(B, Hkv, n, D, generator=g, device=dev, dtype=torch.float16) for _ in range(2))

    def segs(window, new, layout):
        return (_lib.Seg * 2)(_lib.Seg(bits=16, layout=layout, n_tokens=n, pos_base=0, data=window.data_ptr(), slab_tokens=n),
                              _lib.Seg(bits=16, layout=layout, n_tokens=1, pos_base=n, data=new.data_ptr(), slab_tokens=1))

    def step(window, dst, slab):
        ks, vs = segs(kw, k, _lib.LAYOUT_TOKEN_MAJOR), segs(window, v, 0)
        spare = torch.empty(B, Hkv, 1, D, dtype=torch.float16, device=dev)
        w, o = torch.empty(B, Hq, 1, n + 1, dtype=torch.float16, device=dev), torch.empty(B, Hq, 1, D, dtype=torch.float16, device=dev)
        ws = torch.empty(lib.hqekv_decode_workspace_bytes(ks, 2, vs, 2, B, Hq, Hkv, D), dtype=torch.uint8, device=dev)
        x = _lib.StepExtra(append_rows=1, new_k=k.data_ptr(), new_v=v.data_ptr(), k_dst=spare.data_ptr(), v_dst=dst.data_ptr(), k_dst_slab_tokens=1,
                           v_dst_slab_tokens=slab)
        form = lib.hqekv_selftest_step_form(ks, 2, vs, 2, o.data_ptr(), B, Hq, Hkv, D, n + 1, _lib.FUSE_SOFTMAX, ctypes.byref(x))
        rc = lib.hqekv_decode_step(ks, 2, vs, 2, q.data_ptr(), None, 0, w.data_ptr(), o.data_ptr(), B, Hq, Hkv, D, n + 1, ws.data_ptr(), ws.numel(),
                                   _lib.FUSE_SOFTMAX, torch.cuda.current_stream().cuda_stream, ctypes.byref(x))
        assert rc == 0, lib.hqekv_last_error()
        assert torch.equal(spare, k)
        return form, w, o

    elsewhere = torch.empty_like(v)
    form, w0, o0 = step(vw, elsewhere, 1)
    assert form == 1 and torch.equal(elsewhere, v)
    for _ in range(4):
        window = vw.clone()
        form, w, o = step(window, window, n)
        assert form == 2 and torch.equal(w, w0) and torch.equal(o, o0)
        assert torch.equal(window[:, :, :1], v) and torch.equal(window[:, :, 1:], vw[:, :, 1:])


RING = [(1, 8, 8, 300), (8, 32, 8, 300), (9, 32, 8, 300), (8, 40, 8, 300), (2, 72, 9, 200), (1, 4, 1, 3)]   # the last four past what p.V's workgroups cover


def _ring_step(B, Hq, Hkv, n, line, segs):
    from hqekv_amd import _lib
    x = _lib.StepExtra(ring_line=line, ring_order=1)
    return x, _lib.load().hqekv_selftest_step_form(segs[0], 1, segs[1], 1, ctypes.c_void_p(1 << 40), B, Hq, Hkv, D, n, _lib.FUSE_SOFTMAX, ctypes.byref(x))


def _dense(n, k, v):
    from hqekv_amd import _lib
    return ((_lib.Seg * 1)(_lib.Seg(bits=16, layout=_lib.LAYOUT_TOKEN_MAJOR, n_tokens=n, data=k)), (_lib.Seg * 1)(_lib.Seg(bits=16, n_tokens=n, data=v)))


def test_ring_rows_past_what_rides():
    for i, (B, Hq, Hkv, n) in enumerate(RING):
        assert _ring_step(B, Hq, Hkv, n, 1 << 36, _dense(n, 1 << 42, 1 << 43))[1] == (1 if i < 2 else 2)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,n", RING)
def test_a_step_and_the_separate_calls(dev, B, Hq, Hkv, n):
    """Bit for bit: probabilities and output with a ring row beside them and without, the ring row of the one call and of its own."""
    from hqekv_amd import _lib
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev).manual_seed(n + B)
    q, k, v = (torch.randn(B, h, t, D, generator=g, device=dev, dtype=torch.float16) for h, t in ((Hq, 1), (Hkv, n), (Hkv, n)))
    segs = _dense(n, k.data_ptr(), v.data_ptr())
    ws = torch.empty(lib.hqekv_decode_workspace_bytes(segs[0], 1, segs[1], 1, B, Hq, Hkv, D), dtype=torch.uint8, device=dev)
    lines = torch.full((2, n + 2), float("nan"), dtype=torch.float16, device=dev)
    got = []
    for step in (True, False):
        w, o = torch.empty(B, Hq, n, dtype=torch.float16, device=dev), torch.empty(B, Hq, D, dtype=torch.float16, device=dev)
        x, form = _ring_step(B, Hq, Hkv, n, lines.data_ptr(), segs)
        assert form > 0
        rc = lib.hqekv_decode_step(segs[0], 1, segs[1], 1, q.data_ptr(), None, 0, w.data_ptr(), o.data_ptr(), B, Hq, Hkv, D, n, ws.data_ptr(), ws.numel(),
                                   _lib.FUSE_SOFTMAX, st, ctypes.byref(x) if step else None)
        assert rc == 0, lib.hqekv_last_error()
        got.append((w, o))
    assert lib.hqekv_ring_row(got[1][0].data_ptr(), B, Hq, n, lines[1].data_ptr(), 1, st) == 0
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert torch.equal(lines[0, :n], lines[1, :n]) and bool(lines[:, n:].isnan().all()) and bool(lines[:, :n].isfinite().all())


def test_lines_of_the_other_rules():
    """The calls of the kernels' own tests lie on both sides of every line (those tests ask for the form they take)."""
    from hqekv_amd import _lib
    form = _lib.load().hqekv_selftest_form
    assert [form(0, 128 * w, 1, 0) for w in (1, 320, 321, 400, 401, 1500, 1501)] == [21, 21, 121, 121, 112, 112, 11]
    assert [form(1, n, 0, 0) for n in (1, 524287, 524288)] == [1, 1, 4]
    for bits in (1, 2, 4, 8):
        assert [form(2, g, n, bits) for g, n in ((4, 1), (5, 1), (8, 2047 // max(bits, 2)), (8, 2048 // max(bits, 2)))] == [1, 0, 0, 1]
    assert [form(3, r, u, 0) for r, u in ((95, 40), (95, 41), (96, 41))] == [32, 8, 32]
    assert form(9, 1, 1, 1) < 0


@pytest.mark.gpu
@pytest.mark.parametrize("window", [False, True])
def test_replays_of_a_launch_of_its_own(dev, window):
    """Captured into a graph: a ring row past what rides along, a sliding window's row; eager calls between the replays."""
    from hqekv_amd import _lib
    lib, B, Hq, Hkv, n = _lib.load(), 9, 32, 8, 300
    g = torch.Generator(device=dev).manual_seed(8)
    q, k, v, new = (torch.randn(B, h, t, D, generator=g, device=dev, dtype=torch.float16) for h, t in ((Hq, 1), (Hkv, n), (Hkv, n), (Hkv, 1)))
    kept, spare = v.clone(), torch.empty_like(new)
    segs = _dense(n, k.data_ptr(), v.data_ptr())
    ws = torch.empty(lib.hqekv_decode_workspace_bytes(segs[0], 1, segs[1], 1, B, Hq, Hkv, D), dtype=torch.uint8, device=dev)
    line, w, o = (torch.empty(s, dtype=torch.float16, device=dev) for s in ((n,), (B, Hq, n), (B, Hq, D)))
    x = _append(spare.data_ptr(), v.data_ptr(), 1, n) if window else _lib.StepExtra(ring_line=line.data_ptr(), ring_order=1)
    if window:
        x.new_k = x.new_v = new.data_ptr()
    assert lib.hqekv_selftest_step_form(segs[0], 1, segs[1], 1, o.data_ptr(), B, Hq, Hkv, D, n, _lib.FUSE_SOFTMAX, ctypes.byref(x)) == 2

    def step():
        rc = lib.hqekv_decode_step(segs[0], 1, segs[1], 1, q.data_ptr(), None, 0, w.data_ptr(), o.data_ptr(), B, Hq, Hkv, D, n, ws.data_ptr(), ws.numel(),
                                   _lib.FUSE_SOFTMAX, torch.cuda.current_stream().cuda_stream, ctypes.byref(x))
        assert rc == 0, lib.hqekv_last_error()

    def result(run):
        v.copy_(kept)
        for t in (line, w, o, spare):
            t.fill_(7)
        run()
        torch.cuda.synchronize()
        return [t.clone() for t in (line, w, o, v, spare)]

    want = result(step)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        step()
    for _ in range(3):
        assert all(torch.equal(a, b) for a, b in zip(result(graph.replay), want))
        assert all(torch.equal(a, b) for a, b in zip(result(step), want))
    assert torch.equal(want[3][:, :, :1], new if window else kept[:, :, :1]) and torch.equal(want[3][:, :, 1:], kept[:, :, 1:])
