"""The last rows of prompts up to 512 keys in one launch (csrc/prompt_attn.hip, prompt_last_short_kernel): both sides of
every number of waves, column tiles that end inside a head, one row and 32, masks, q and k as slices of a fused projection;
513 keys for the form beyond."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 20, 33, 64, 65, 128, 129, 250, 256, 257, 511, 512, 513])
@pytest.mark.parametrize("B,Hq,Hkv,R", [(1, 32, 8, 20), (2, 7, 1, 32), (3, 5, 5, 1), (1, 24, 8, 13)])
@pytest.mark.parametrize("masked", [False, True])
def test_against_the_fp16_chain(dev, T, B, Hq, Hkv, R, masked):
    """Tolerance: three roundings of a logit may fall to the other half -- the product's, 2^-5 below 64 and times the scale 2.8e-3,
    the scaled one's and the masked one's, 2^-8 each below 8 -- and move its probability by as much of itself, and the
    probability's own, 2^-11: 1.1e-2."""
    from hqekv_amd import _lib
    from hqekv_amd.prompt_attention import prompt_last_rows
    R = min(R, T)
    assert (_lib.load().hqekv_prompt_last_rows_workspace_bytes(B, Hq, T) == 0) == (T <= 512)   # (the form of one launch needs none)
    g = torch.Generator(device=dev).manual_seed(T * 7 + Hq)
    fused = torch.randn(B, T, (Hq + Hkv) * 128, generator=g, device=dev, dtype=torch.float16)
    q = fused[..., :Hq * 128].view(B, T, Hq, 128).transpose(1, 2)
    k = fused[..., Hq * 128:].view(B, T, Hkv, 128).transpose(1, 2)
    mask = None
    causal = torch.full((T, T), -65504.0, device=dev).triu(1).half()[T - R:].expand(B, 1, R, T)
    if masked:
        mask = causal.clone()
        mask[..., ::3] = torch.randn(B, 1, R, len(range(0, T, 3)), generator=g, device=dev).half()
    got = prompt_last_rows(q, k, 128 ** -0.5, R, None if mask is None else torch.cat([torch.zeros(B, 1, T - R, T, device=dev).half(), mask], 2))
    heads = k.float().repeat_interleave(Hq // Hkv, 1)
    s = torch.matmul(q[:, :, T - R:].float(), heads.transpose(2, 3).contiguous()).half()
    s = (s.float() * 128 ** -0.5).half()
    s = (s.float() + (causal if mask is None else mask).float()).half().float().clamp_min(-65504.0)
    want = s.softmax(-1)
    assert got.shape == want.shape and torch.isfinite(got).all()
    torch.testing.assert_close(got.float(), want, rtol=1.1e-2, atol=1e-6)
    assert (got.float().sum(-1) - 1).abs().max() < 2e-2
