"""Which form of the prompt kernel a call takes (csrc/prompt_attn.hip, prompt_form), on both sides of its lines: numbers of
workgroups at which the second 256 come reversed whole, in part and by eights, rows and keys that end inside a step."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,T,form", [
    (1, 100, 100, 450, 121), (1, 101, 101, 450, 112),              # 400 and 404 workgroups of 128 rows
    (2, 64, 8, 385, 112), (4, 32, 8, 511, 112),                    # 512: by eights
    (1, 70, 10, 1024, 112), (1, 96, 24, 700, 112),                 # 560, 576
    (1, 64, 8, 640, 21), (1, 64, 8, 641, 121),                     # 640 and 704 of 64 rows
    (3, 125, 25, 512, 112), (4, 94, 47, 449, 11)])                 # 1500 and 1504
def test_on_both_sides_of_the_lines(dev, B, Hq, Hkv, T, form, causal):
    """Tolerance: probabilities are rounded to fp16 (2^-11) before the second product and the output once more."""
    from hqekv_amd import _lib
    from hqekv_amd.prompt_attention import prompt_attention
    assert _lib.load().hqekv_selftest_form(0, T, B * Hq, 0) == form
    g = torch.Generator(device=dev).manual_seed(T + Hq)
    q, k, v = (torch.randn(B, h, T, 128, generator=g, device=dev, dtype=torch.float16) for h in (Hq, Hkv, Hkv))
    out = prompt_attention(q, k, v, 128 ** -0.5, causal=causal)
    for h in sorted({0, 1, 7, 8, Hq // 2, Hq - 1}):
        s = q[:, h].float() @ k[:, h // (Hq // Hkv)].float().transpose(1, 2).contiguous() * 128 ** -0.5
        if causal:
            s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=dev).triu(1), float("-inf"))
        ref = s.softmax(-1) @ v[:, h // (Hq // Hkv)].float()
        got = out[:, h] if out.shape[1] == Hq else out.transpose(1, 2)[:, h]
        torch.testing.assert_close(got.float(), ref, rtol=2e-3, atol=2e-3)
