"""p.V of five to eight query heads per KV head on both sides of the line between one block per workgroup and several
(six workgroups per CU): a class that ends on the line, one that is 32 tokens over it, two classes of which one ends inside
a workgroup's run.  Against the CPU oracle, at the tolerances of test_tiles_gpu.py; the outputs also by what their
probabilities differ: where one logit of the three million here rounds to the other neighbouring half, its probability moves
by up to ulp(logit) of itself, within the probabilities' tolerance, and the output by that times at most the largest value
of V (dequantised values lie within their group's range)."""
import pytest
import torch

from hqekv_amd import synth
from oracle import hqe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rep", [5, 8])
@pytest.mark.parametrize("classes,rows", [({4: 64}, 8), ({4: 65}, 3), ({2: 33, 8: 17}, 4)], ids=["resident", "over", "two"])
def test_line_between_forms(dev, n_rep, classes, rows):
    from hqekv_amd import _lib
    from hqekv_amd.attention import DecodePlan, decode_attention
    B, Hkv, D, n = 24, 8, 128, 32 * sum(classes.values())
    q, K, V = synth.make_qkv(B, n_rep * Hkv, Hkv, n, D, 9)
    tokens, at = {b: torch.arange(0) for b in (16, 8, 4, 2, 1)}, 0
    for bits, c in classes.items():
        tokens[bits] = torch.arange(at, at + 32 * c)
        at += 32 * c
    cache = synth.build_cache(K, V, tokens, 0, O.uniform_group_quantize_pack_last_dim)
    w_ref, o_ref = O.qkv_matmul(q, cache, None, D, use_mask=False, round_per_class=False)
    plan = DecodePlan(q.to(dev), synth.cache_to(cache, dev))
    assert _lib.load().hqekv_pv_workspace_bytes(plan.v_segs, plan.n_v, B, n_rep * Hkv, Hkv, D) == rows * B * n_rep * Hkv * 512   # blocks: 8, 9, 5 + 5
    w, o = decode_attention(q.to(dev), synth.cache_to(cache, dev), None, n, zero_init=False, flags=1)
    torch.testing.assert_close(w.float().cpu(), w_ref.float(), rtol=1e-3, atol=2e-3)
    moved = (w.float().cpu() - w_ref.float()).abs().sum(-1, keepdim=True) * V.float().abs().max()
    off = (o.float().cpu() - o_ref.float()).abs() - 1e-3 * o_ref.float().abs() - 2e-3 - moved
    assert off.max() <= 0, (off.max(), moved.max())
