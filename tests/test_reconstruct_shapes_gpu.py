"""The reconstruction's turned tiles (csrc/reconstruct.hip): head sizes below, at and past 128 channels, classes that end inside
a 32-token group, a tile or a half of it, fp16 K rows of every length modulo eight -- against the oracle's dequantiser."""
import pytest
import torch

from hqekv_amd import synth
from oracle import hqe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 96, 128, 160, 256])
@pytest.mark.parametrize("blocks,residual", [((1, 1, 1, 1, 1), 5), ((5, 3, 4, 6, 2), 0), ((4, 8, 0, 9, 1), 33), ((0, 5, 7, 0, 0), 1)])
def test_shapes(dev, D, blocks, residual):
    from hqekv_amd.hqe_2 import KV_cache_reconstruct_hqe
    B, H, n = 2, 3, 32 * sum(blocks)
    _, K, V = synth.make_qkv(B, H, H, n + residual, D, D + n)
    order = torch.randperm(n // 32, generator=torch.Generator().manual_seed(n))
    classes, at = {}, 0
    for bits, c in zip((16, 8, 4, 2, 1), blocks):
        classes[bits] = (order[at:at + c].sort()[0][:, None] * 32 + torch.arange(32)).reshape(-1)
        at += c
    cache = synth.build_cache(K, V, classes, residual, O.uniform_group_quantize_pack_last_dim)
    want = O.reconstruct_cache(cache, "uniform_group")
    got = KV_cache_reconstruct_hqe(synth.cache_to(cache, dev), "uniform_group")
    if blocks[0] and D == 128:   # fp16 classes of ragged length on both sides
        cut = 32 * blocks[0] - 13
        cache = (cache[0][..., :cut].contiguous(), cache[1][:cut].contiguous(), cache[2][:, :, :cut].contiguous(), cache[3][:cut].contiguous(), *cache[4:])
        want = (*want, *O.reconstruct_cache(cache, "uniform_group"))
        got = (*got, *KV_cache_reconstruct_hqe(synth.cache_to(cache, dev), "uniform_group"))
    for g, w in zip(got, want):
        assert torch.equal(g.cpu().view(torch.int16), w.contiguous().view(torch.int16))
