"""A hybrid cache back into dense K and V in one launch against the oracle's class-by-class restoration, bit for bit."""
import pytest
import torch

from hqekv_amd import synth
from oracle import hqe_oracle as O

pytestmark = pytest.mark.gpu
LOW_NORMAL = "high_uniform_group_low_normal_group"


def _cache(dev, B, H, T, D, residual, fractions, strategy, seed=5):
    from hqekv_amd import pack_unpack as PU

    def quantize(x, group, bits):
        if bits == 1 and strategy == LOW_NORMAL:
            return PU.normal_group_quantize_pack_last_dim(x, group, 1)
        return PU.uniform_group_quantize_pack_last_dim(x, group, bits)
    _, K, V = synth.make_qkv(B, H, H, T + residual, D, seed, dev)
    return synth.build_cache(K, V, synth.split_blocks(T, fractions, seed), residual, quantize)


def _check(pkv, strategy):
    from hqekv_amd.hqe_2 import KV_cache_reconstruct_hqe
    got = KV_cache_reconstruct_hqe(pkv, strategy)
    want = O.reconstruct_cache(synth.cache_to(pkv, "cpu"), strategy)
    for g, w, side in zip(got, want, "KV"):
        assert torch.equal(g.cpu().view(torch.int16), w.contiguous().view(torch.int16)), side


@pytest.mark.parametrize("strategy", ["uniform_group", LOW_NORMAL])
@pytest.mark.parametrize("B,H,T,D,residual,fractions", [
    (1, 1, 32, 128, 0, (0, 0, 0, 1, 0, 0)),                      # one group of one class
    (2, 3, 1056, 128, 17, (.1, .2, .2, .2, .2, .1)),             # every class, ragged tiles, a residual
    (1, 2, 4096, 128, 63, (.05, .15, .3, .2, .1, .2)),
    (1, 2, 416, 64, 1, (.2, .2, .2, .2, .1, .1)),                # other head sizes: half a channel tile, one and a half
    (1, 2, 416, 192, 3, (.2, .2, .2, .2, .1, .1)),
])
def test_every_class(dev, B, H, T, D, residual, fractions, strategy):
    _check(_cache(dev, B, H, T, D, residual, fractions, strategy), strategy)


def test_positions_nobody_names_are_zero(dev):
    """kv_seq_len beyond the kept tokens (it counts evicted ones), an absent side, a class of a ragged token count."""
    pkv = _cache(dev, 1, 2, 512, 128, 5, (.2, .2, .2, .2, .2), "uniform_group")
    _check(pkv[:41] + (pkv[41] + 100,), "uniform_group")
    ragged = list(pkv)
    ragged[0], ragged[1] = pkv[0][..., :45].contiguous(), pkv[1][:45].contiguous()
    ragged[2], ragged[3] = pkv[2][:, :, :45].contiguous(), pkv[3][:45].contiguous()
    _check(tuple(ragged), "uniform_group")
    ragged[4:8] = [None] * 4
    _check(tuple(ragged), "uniform_group")


@pytest.mark.parametrize("n", [1, 31, 32, 257, 5000])
def test_cover_check(dev, n):
    from hqekv_amd.attention import idx_cover_once
    p = torch.randperm(n, generator=torch.Generator().manual_seed(n))
    cut = n // 3

    def parts(x):
        return [t for t in (x[:cut].to(dev), x[cut:].to(dev)) if t.numel()]
    assert idx_cover_once(parts(p), n)
    for bad in (-1, n, int(p[-1])):
        q = p.clone()
        q[0] = bad
        assert idx_cover_once(parts(q), n) == (bad == int(p[0]))


def test_more_tiles_than_a_grid_dimension_holds(dev):
    """4.2 million tokens per side: 66000 tiles of 128 for both."""
    from hqekv_amd import pack_unpack as PU
    from hqekv_amd.hqe_2 import KV_cache_reconstruct_hqe
    T, D = 32 * 132000, 32
    g = torch.Generator(device=dev).manual_seed(3)
    kc = torch.randint(-2 ** 31, 2 ** 31 - 1, (1, 1, D, T // 16), generator=g, device=dev, dtype=torch.int32)
    vc = torch.randint(-2 ** 31, 2 ** 31 - 1, (1, 1, T, D // 16), generator=g, device=dev, dtype=torch.int32)
    ks, kz = (torch.randn(1, 1, D, T // 32, generator=g, device=dev).half() for _ in range(2))
    vs, vz = (torch.randn(1, 1, T, 1, generator=g, device=dev).half() for _ in range(2))
    idx = torch.arange(T, device=dev)
    pkv = [None] * 42
    pkv[20:24] = kc, idx, ks, kz
    pkv[24:28] = vc, idx.clone(), vs, vz
    pkv[41] = T
    K, V = KV_cache_reconstruct_hqe(tuple(pkv), "uniform_group")
    assert torch.equal(V, PU.uniform_group_dequantize_unpack_last_dim(vc, vs, vz, 32, 2))
    assert torch.equal(K, PU.uniform_group_dequantize_unpack_last_dim(kc, ks, kz, 32, 2).transpose(2, 3))


@pytest.mark.parametrize("slots", [(0,), ("transposed", 0), (2,), (39, 40), ("window", 39, 40)])
def test_fp16_planes_at_any_element(dev, slots):
    """Planes that start at an odd element: dense, K as the transposed view of token-major rows, heads of longer buffers."""
    pkv = list(_cache(dev, 1, 2, 512, 128, 5, (.2, .2, .2, .2, .2), "uniform_group"))
    for s in slots[isinstance(slots[0], str):]:
        x = pkv[s].transpose(2, 3) if slots[0] == "transposed" else pkv[s]
        rows = x.shape[2] + (3 if slots[0] == "window" else 0)
        room = torch.empty(x.numel() // x.shape[2] * rows + 1, dtype=torch.float16, device=dev)[1:]
        room = room.view(*x.shape[:2], rows, x.shape[3])[:, :, :x.shape[2]].copy_(x)
        pkv[s] = room.transpose(2, 3) if slots[0] == "transposed" else room
        assert pkv[s].data_ptr() % 16 == 2
    _check(tuple(pkv), "uniform_group")


def test_head_size_beyond_the_kernel(dev):
    _check(_cache(dev, 1, 1, 64, 4128, 3, (.5, 0, 0, .5, 0), "uniform_group"), "uniform_group")


def test_positions_outside_the_cache(dev):
    """One that counts from the end is taken, as an index into a tensor is; one that names no row is an error."""
    from hqekv_amd.hqe_2 import KV_cache_reconstruct_hqe
    pkv = list(_cache(dev, 1, 2, 512, 128, 5, (.2, .2, .2, .2, .2), "uniform_group"))
    T = pkv[41]
    pkv[1] = pkv[1] - T
    _check(tuple(pkv), "uniform_group")
    for slot, bad in ((3, T), (13, -T - 1), (25, 2 ** 40)):
        wrong = list(pkv)
        wrong[slot] = pkv[slot].clone()
        wrong[slot][-1] = bad
        with pytest.raises(IndexError):
            KV_cache_reconstruct_hqe(tuple(wrong), "uniform_group")
    with pytest.raises(ValueError):
        KV_cache_reconstruct_hqe(tuple(pkv[:41]) + (3,), "uniform_group")   # fewer positions than the residual has rows


@pytest.mark.parametrize("seen", [False, True])
def test_reconstruction_captured_into_a_graph(dev, seen):
    """Positions never looked at before (class by class) or known to cover the cache (one launch): every replay gives what
    the eager call gives, on the cache's contents of the time."""
    from hqekv_amd.hqe_2 import KV_cache_reconstruct_hqe
    pkv = _cache(dev, 1, 2, 512, 128, 5, (.2, .2, .2, .2, .2), "uniform_group")
    if seen:
        KV_cache_reconstruct_hqe(pkv, "uniform_group")
    warm = _cache(dev, 1, 2, 512, 128, 5, (.2, .2, .2, .2, .2), "uniform_group")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        KV_cache_reconstruct_hqe(warm, "uniform_group")
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = KV_cache_reconstruct_hqe(pkv, "uniform_group")
    torch.cuda.synchronize()
    want = O.reconstruct_cache(synth.cache_to(pkv, "cpu"), "uniform_group")
    for turn in range(4):
        for g in got:
            g.fill_(turn)
        graph.replay()
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            assert torch.equal(g.cpu().view(torch.int16), w.contiguous().view(torch.int16)), turn
        pkv[2].neg_()
        want = O.reconstruct_cache(synth.cache_to(pkv, "cpu"), "uniform_group")


def test_positions_as_any_integers_anywhere(dev):
    """Positions as 32-bit numbers, on the host, as every other element of a longer array: what indexing a tensor takes."""
    pkv = list(_cache(dev, 1, 2, 512, 128, 5, (.2, .2, .2, .2, .2), "uniform_group"))
    pkv[1], pkv[5], pkv[9] = pkv[1].cpu(), pkv[5].to(torch.int32), pkv[9].repeat_interleave(2)[::2]
    _check(tuple(pkv), "uniform_group")
    pkv[1] = pkv[1] - pkv[41]                    # counted from the end, as well
    _check(tuple(pkv), "uniform_group")
