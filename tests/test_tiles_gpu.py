"""The matrix-core launches of a decode step (csrc/decode_qk.hip, decode_pv.hip) at the edges of their tiles, against the
CPU oracle: classes of a few blocks up to one more than a tile, every count of query heads per KV head they pad (1 to 16),
positions in runs and shuffled, residuals of odd and even length, and a launch of several blocks per workgroup."""
import pytest
import torch

from hqekv_amd import synth
from oracle import hqe_oracle as O

pytestmark = pytest.mark.gpu
RTOL, ATOL = 1e-3, 2e-3


def _quant(low_normal):
    def f(x, g, bits):
        if bits == 1 and low_normal:
            return O.normal_group_quantize_pack_last_dim(x, 32, 1)
        return O.uniform_group_quantize_pack_last_dim(x, 32, bits)
    return f


@pytest.mark.parametrize("blocks", [(1, 1, 1, 1, 1), (4, 7, 8, 9, 8), (5, 9, 16, 17, 1), (0, 4, 0, 33, 7)],
                         ids=lambda b: "-".join(map(str, b)))
@pytest.mark.parametrize("n_rep,B,residual,low_normal,fused", [
    (1, 2, 0, False, True), (3, 1, 1, False, True), (4, 1, 64, True, True), (4, 3, 65, False, False),
    (5, 2, 16, False, True), (8, 1, 31, True, True), (12, 1, 2, False, True), (16, 1, 0, False, False)])
@pytest.mark.parametrize("shuffled", [False, True], ids=["runs", "shuffled"])
def test_tile_edges(dev, blocks, n_rep, B, residual, low_normal, fused, shuffled):
    from hqekv_amd.attention import decode_attention
    Hkv, D, n = 2, 128, 32 * sum(blocks)
    q, K, V = synth.make_qkv(B, n_rep * Hkv, Hkv, n + residual, D, 77)
    order = torch.randperm(n // 32, generator=torch.Generator().manual_seed(n))
    classes, at = {}, 0
    for bits, c in zip((16, 8, 4, 2, 1), blocks):
        classes[bits] = (order[at:at + c].sort()[0][:, None] * 32 + torch.arange(32)).reshape(-1)
        at += c
    override = None
    if shuffled:
        perm, override, at = torch.randperm(n, generator=torch.Generator().manual_seed(n + 1)), {}, 0
        for bits, tok in classes.items():
            override[bits] = perm[at:at + tok.numel()]
            at += tok.numel()
    cache = synth.build_cache(K, V, classes, residual, _quant(low_normal), override)
    strategy = "high_uniform_group_low_normal_group" if low_normal else "uniform_group"
    w_ref, o_ref = O.qkv_matmul(q, cache, None, D, strategy, use_mask=False, round_per_class=False)
    w, o = decode_attention(q.to(dev), synth.cache_to(cache, dev), None, n + residual, zero_init=False, flags=1 if fused else 0,
                            low_uniform=not low_normal)
    torch.testing.assert_close(w.float().cpu(), w_ref.float(), rtol=RTOL, atol=ATOL)
    torch.testing.assert_close(o.float().cpu(), o_ref.float(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("n_rep", [4, 5, 12])
def test_several_blocks_per_workgroup(dev, n_rep):
    """More blocks of V than workgroups fit on the chip: the looping form, with every class and a ragged last round."""
    from hqekv_amd.attention import decode_attention
    B, Hkv, D, residual = 20, 8, 128, 13
    q, K, V = synth.make_qkv(B, n_rep * Hkv, Hkv, 3200 + residual, D, 5)
    classes = synth.split_blocks(3200, (0.1, 0.2, 0.3, 0.3, 0.1), 5)
    cache = synth.build_cache(K, V, classes, residual, O.uniform_group_quantize_pack_last_dim)
    w_ref, o_ref = O.qkv_matmul(q, cache, None, D, use_mask=False, round_per_class=False)
    w, o = decode_attention(q.to(dev), synth.cache_to(cache, dev), None, int(cache[41]), zero_init=False, flags=1)
    torch.testing.assert_close(w.float().cpu(), w_ref.float(), rtol=RTOL, atol=ATOL)
    torch.testing.assert_close(o.float().cpu(), o_ref.float(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("n_rep,low_normal,shuffled,B", [(4, False, False, 512), (5, True, False, 512), (4, True, True, 512), (3, False, False, 300), (12, False, False, 512)])
def test_several_tiles_per_workgroup_of_scores(dev, n_rep, low_normal, shuffled, B):
    """A launch long enough for q.K^T to take four tiles per workgroup -- classes that end inside a wave's tile, inside a
    workgroup's four, exactly at their end -- against the same rows in a batch of two, which takes one tile each."""
    from hqekv_amd.attention import decode_attention
    from hqekv_amd.pack_unpack import normal_group_quantize_pack_last_dim, uniform_group_quantize_pack_last_dim
    blocks, residual, Hkv, D = (5, 9, 33, 31, 33), 65, 2, 128
    n = 32 * sum(blocks)

    def quantize(x, g, bits):
        return normal_group_quantize_pack_last_dim(x, 32, 1) if bits == 1 and low_normal else uniform_group_quantize_pack_last_dim(x, 32, bits)
    q, K, V = synth.make_qkv(2, n_rep * Hkv, Hkv, n + residual, D, 78, dev)
    order = torch.randperm(n if shuffled else n // 32, generator=torch.Generator().manual_seed(n))
    tokens = order if shuffled else (order[:, None] * 32 + torch.arange(32)).reshape(-1)
    classes, at = {}, 0
    for bits, c in zip((16, 8, 4, 2, 1), blocks):
        classes[bits] = tokens[at:at + 32 * c].sort()[0]
        at += 32 * c
    pkv = synth.build_cache(K, V, classes, residual, quantize)
    big = tuple(x.repeat(B // 2, 1, 1, 1) if torch.is_tensor(x) and x.dim() == 4 else x for x in pkv)
    small = decode_attention(q, pkv, None, n + residual, True, low_uniform=not low_normal)
    got = decode_attention(q.repeat(B // 2, 1, 1, 1), big, None, n + residual, True, low_uniform=not low_normal)
    for g, w in zip(got, small):
        torch.testing.assert_close(g.float(), w.repeat(B // 2, 1, 1, 1).float(), rtol=2e-3, atol=1e-3)


@pytest.mark.parametrize("n_rep", [1, 4, 5, 12])
@pytest.mark.parametrize("B,tiling", [(1, 0), (400, 0), (1, 1), (1, 3)], ids=["one-tile", "four-tiles", "8waves", "wave512"])
def test_a_score_of_minus_infinity_has_probability_zero(dev, n_rep, B, tiling):
    """A finite key whose score leaves fp16's range on the negative side, alone in its lane, its tile or its class."""
    from hqekv_amd import _lib
    from hqekv_amd.attention import decode_attention
    Hkv, D, blocks, residual = 2, 128, (4, 8, 8, 8, 8), 65
    n = 32 * sum(blocks)
    q, K, V = synth.make_qkv(1, Hkv, Hkv, n + residual, D, 43)
    far = [0, 1, 2, 3, 40, *range(n, n + 8), n + 64]   # (the residual's last token is alone in its tile)
    K[:, :, far] = (-30000.0 * q.sign()).half()   # scores of -30000 |q|_1: three million
    far += list(range(32 * 4, 32 * 12))           # and a whole class: tiles without a finite score
    K[:, :, 32 * 4:32 * 12] = (-30000.0 * q.sign()).half()
    classes, at = {}, 0
    for bits, c in zip((16, 8, 4, 2, 1), blocks):
        classes[bits] = torch.arange(32 * at, 32 * (at + c))
        at += c
    q = q.repeat_interleave(n_rep, 1)
    pkv = synth.build_cache(K, V, classes, residual, O.uniform_group_quantize_pack_last_dim)
    w_ref, o_ref = O.qkv_matmul(q, pkv, None, D, use_mask=False, round_per_class=False)
    big = tuple(x.repeat(B, 1, 1, 1) if torch.is_tensor(x) and x.dim() == 4 else x for x in synth.cache_to(pkv, dev))
    w, o = decode_attention(q.to(dev).repeat(B, 1, 1, 1), big, None, n + residual, zero_init=False, flags=1 | _lib.qk_tiling(tiling))
    assert not w[..., far].any()
    torch.testing.assert_close(w[-1:].float().cpu(), w_ref.float(), rtol=RTOL, atol=ATOL)
    torch.testing.assert_close(o[-1:].float().cpu(), o_ref.float(), rtol=RTOL, atol=ATOL)


def _bad_cache(n_rep, value):
    """Every class and a residual, some keys of each not finite: an element of the fp16 rows, the scale of a quantised group."""
    Hkv, D, blocks, residual = 2, 128, (5, 9, 9, 9, 9), 33
    n = 32 * sum(blocks)
    q, K, V = synth.make_qkv(1, n_rep * Hkv, Hkv, n + residual, D, 41)
    classes, at = {}, 0
    for bits, c in zip((16, 8, 4, 2, 1), blocks):
        classes[bits] = torch.arange(32 * at, 32 * (at + c))
        at += c
    pkv = synth.build_cache(K, V, classes, residual, O.uniform_group_quantize_pack_last_dim)
    for h, d, t in ((0, 3, 0), (0, 70, 37), (1, 127, 159)):
        pkv[0][0, h, d, t] = value                      # fp16 class (B, H, D, T)
    for h, t, d in ((0, 3, 9), (1, 0, 64), (1, 32, 5)):   # (32: the last one, which the unused rows of its tile repeat)
        pkv[39][0, h, t, d] = value                     # residual (B, H, T, D)
    for base in (4, 12, 20, 28):
        pkv[base + 2][0, 0, 17, 0] = value              # a group's scale
        pkv[base + 2][0, 1, 99, 8] = value
    return q, pkv


@pytest.mark.parametrize("n_rep", [1, 4, 5, 12])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("B", [1, 400], ids=["one-tile", "four-tiles"])
def test_a_key_that_is_not_finite_stays_with_its_token(dev, n_rep, value, B):
    """Raw scores: infinities and NaN exactly where the definition has them, every other token's score as it is."""
    from hqekv_amd.attention import DecodePlan
    q, pkv = _bad_cache(n_rep, value)
    K = O.reconstruct_cache(pkv, "uniform_group")[0]
    want = (q.view(1, 2, n_rep, 1, 128).double() * K[:, :, None].double()).sum(-1).view(1, 2 * n_rep, 1, -1)
    big = tuple(x.repeat(B, 1, 1, 1) if torch.is_tensor(x) and x.dim() == 4 else x for x in synth.cache_to(pkv, dev))
    plan = DecodePlan(q.to(dev).repeat(B, 1, 1, 1), big)
    plan.run_qk(q.to(dev).repeat(B, 1, 1, 1))
    got = plan.weights.cpu()
    assert torch.equal(got.view(torch.int16), got[:1].expand_as(got).contiguous().view(torch.int16))
    # scores are a few hundred at the most, rounded to fp16 once; fp32 sums of 128 products move them by a place
    torch.testing.assert_close(got[:1].double(), want.half().double(), rtol=2e-3, atol=2e-3, equal_nan=True)


@pytest.mark.parametrize("n_rep", [4, 5])
def test_a_masked_slot_that_holds_no_number(dev, n_rep):
    """Slots whose keys are NaN, masked out: the probabilities of all others are what they are without them."""
    from hqekv_amd.attention import decode_attention
    q, pkv = _bad_cache(n_rep, float("nan"))
    pkv = [x.clone() if torch.is_tensor(x) else x for x in pkv]
    bad = torch.isnan(O.reconstruct_cache(tuple(pkv), "uniform_group")[0]).any(-1).any(0).any(0)
    mask = torch.zeros(1, 1, 1, int(pkv[41]), dtype=torch.float16)
    mask[..., bad] = torch.finfo(torch.float16).min
    w, o = decode_attention(q.to(dev), synth.cache_to(tuple(pkv), dev), mask.to(dev), int(pkv[41]), zero_init=False)
    for i, x in enumerate(pkv[:41]):
        if torch.is_tensor(x) and x.dtype == torch.float16:
            x[torch.isnan(x)] = 0
    w_ref, o_ref = O.qkv_matmul(q, tuple(pkv), mask, 128, round_per_class=False)
    torch.testing.assert_close(w.float().cpu(), w_ref.float(), rtol=RTOL, atol=ATOL)
    torch.testing.assert_close(o.float().cpu(), o_ref.float(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("n_rep,residual", [(4, 33), (5, 2), (12, 1)])
@pytest.mark.parametrize("fused", [True, False], ids=["fused", "general"])
def test_a_value_row_that_is_not_finite(dev, n_rep, residual, fused):
    """The last row of every V class holds an infinity (which the unused rows of its block repeat): the outputs are the
    infinities of the definition, not NaN."""
    from hqekv_amd.attention import decode_attention
    Hkv, D, sizes = 2, 128, (45, 33, 31, 70, 5)
    n = sum(sizes)
    g = torch.Generator().manual_seed(3)
    q, K, V = synth.make_qkv(1, n_rep * Hkv, Hkv, n + residual, D, 44)
    q = q * 0.05                                  # (every probability above fp16's smallest)
    pkv = [None] * 42
    pkv[0], pkv[1] = K[:, :, :n].transpose(2, 3).contiguous(), torch.arange(n)   # K: one fp16 class
    perm, at = torch.randperm(n, generator=g), 0
    for bits, slot, c in zip((16, 8, 4, 2, 1), (2, 8, 16, 24, 32), sizes):
        pos = perm[at:at + c]
        rows = V[:, :, pos].contiguous()
        if bits == 16:
            rows[:, :, -1, 7] = float("inf")
            pkv[2], pkv[3] = rows, pos
        else:
            code, scale, zero = O.uniform_group_quantize_pack_last_dim(rows, 32, bits)
            zero[:, :, -1, 2] = float("inf")
            pkv[slot], pkv[slot + 1], pkv[slot + 2], pkv[slot + 3] = code, pos, scale, zero
        at += c
    pkv[39], pkv[40] = K[:, :, n:].contiguous(), V[:, :, n:].contiguous()
    pkv[40][:, :, -1, 20] = float("inf")
    pkv[41] = n + residual
    pkv = tuple(pkv)
    w, o = decode_attention(q.to(dev), synth.cache_to(pkv, dev), None, n + residual, zero_init=False, flags=1 if fused else 0)
    assert float(w.min()) > 0
    dense = O.reconstruct_cache(pkv, "uniform_group")[1].double()
    want = torch.matmul(w.cpu().double().view(1, Hkv, n_rep, -1), dense).view(1, n_rep * Hkv, 1, D)
    assert torch.isinf(want).any()
    torch.testing.assert_close(o.cpu().double(), want.half().double(), rtol=RTOL, atol=ATOL, equal_nan=True)
