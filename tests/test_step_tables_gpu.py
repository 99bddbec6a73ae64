"""A layer's segment tables read in C++ (``_host.step_tables``) against those that ``SegmentMemo.build`` lists in Python:
the same step bit for bit over every form of tuple that either takes -- missing classes, positions in runs and shuffled, fp16
keys as a transposed view, the normal-quantile class --, and the same refusals."""
import ctypes as C

import pytest
import torch

from hqekv_amd import synth
from oracle import hqe_oracle as O

pytestmark = pytest.mark.gpu


def _cache(dev, B, blocks, low_normal=False, shuffled=False):
    n, Hkv, D = 32 * sum(blocks), 2, 128
    _, K, V = synth.make_qkv(B, 8, Hkv, n, D, 3)
    order = torch.randperm(n, generator=torch.Generator().manual_seed(n)) if shuffled else torch.arange(n)
    tokens, at = {}, 0
    for bits, c in zip((16, 8, 4, 2, 1), blocks):
        tokens[bits] = order[at:at + 32 * c]
        at += 32 * c

    def quantize(x, g, bits):
        return O.normal_group_quantize_pack_last_dim(x, 32, 1) if bits == 1 and low_normal else O.uniform_group_quantize_pack_last_dim(x, 32, bits)
    return synth.cache_to(synth.build_cache(K, V, {b: t.sort()[0] for b, t in tokens.items()}, 0, quantize, tokens if shuffled else None), dev), n


def _step(tables, pkv, n, q, k, v):
    buf = [torch.zeros(*k.shape[:2], 64, 128, dtype=torch.float16, device=q.device) for _ in range(2)]
    buf[0][:, :, :3], buf[1][:, :, :3] = k * 0.5, v * 0.25
    ring = torch.zeros(20, n + 8, dtype=torch.float16, device=q.device)
    w, o, _ = tables.step(q, k, v, pkv, *buf, 3, n + 4, ring, 2, n + 4)
    return w, o, ring, *buf


@pytest.mark.parametrize("form", ["all", "transposed keys", "normal", "shuffled", "two", "columns of a wider array"])
def test_same_step(dev, form):
    from hqekv_amd import _lib
    from hqekv_amd.attention import SegmentMemo, decode_attention, idx_cover_once
    B = 2
    blocks = {"two": (0, 0, 5, 9, 0)}.get(form, (3, 2, 5, 7, 4))
    pkv, n = _cache(dev, B, blocks, low_normal=form == "normal", shuffled=form == "shuffled")
    pkv = list(pkv)
    if form == "transposed keys":
        pkv[0] = pkv[0].transpose(2, 3).contiguous().transpose(2, 3)
    plain = form != "columns of a wider array"
    if not plain:   # codes that have to be copied first: only the Python tables take them
        wide = torch.zeros(*pkv[12].shape[:3], pkv[12].shape[3] + 1, dtype=pkv[12].dtype, device=dev)
        wide[..., :-1] = pkv[12]
        pkv[12] = wide[..., :-1]
    pkv = tuple(pkv)
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(B, h, 1, 128, generator=g).half().to(dev) for h in (32, 2, 2))
    low_uniform = form != "normal"
    native = _lib.host().step_tables(q, pkv, low_uniform, idx_cover_once)
    assert (native is not None) == plain
    listed, memo = SegmentMemo(), SegmentMemo()
    listed.build(pkv, q.device, low_uniform)
    assert listed.partition
    want = _step(_lib.host().StepTables(C.addressof(listed.k_arr), listed.n_k, C.addressof(listed.v_arr), listed.n_v), pkv, n, q, k, v)
    got = _step(memo.steps(pkv, q, low_uniform, False), pkv, n, q, k, v)
    assert memo.steps(pkv, q, low_uniform, True) is memo.steps(pkv, q, low_uniform, False)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    # the same memo behind a call that wants the Python tables
    a = decode_attention(q, pkv, None, n, True, low_uniform=low_uniform, memo=memo)
    b = decode_attention(q, pkv, None, n, True, low_uniform=low_uniform, memo=listed)
    assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_refusals(dev):
    from hqekv_amd import _lib
    from hqekv_amd.attention import SegmentMemo, idx_cover_once
    pkv, n = _cache(dev, 2, (3, 2, 5, 7, 4))
    q = torch.zeros(2, 32, 1, 128, dtype=torch.float16, device=dev)
    holes = list(pkv)
    holes[13] = pkv[13].clone()
    holes[13][0] = holes[13][1]   # a position twice, another not at all
    for t in (tuple(holes), (None,) * 42):
        assert _lib.host().step_tables(q, t, True, idx_cover_once) is None
    assert SegmentMemo().steps(tuple(holes), q, True, False) is None
    assert _lib.host().step_tables(q[:1], pkv, True, idx_cover_once) is None   # another batch size
    assert _lib.host().step_tables(q.cpu(), pkv, True, idx_cover_once) is None
