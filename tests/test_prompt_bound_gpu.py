"""The prompt kernel keeps the bound that its exponents are relative to while a larger score holds little of the row's sum
(csrc/prompt_attn.hip): scores that climb along the keys, by less than the slack, by a little more, and by far more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,T", [(1, 4, 97), (1, 8, 700), (2, 40, 1100), (4, 64, 1200)])   # 4 to 2560 workgroups: every form
@pytest.mark.parametrize("climb", [0.01, 0.4, 7.5, 8.5, 60.0])   # powers of two per 32 keys
@pytest.mark.parametrize("down", [False, True])
def test_scores_that_climb(dev, B, Hq, T, climb, down):
    """Tolerance: a weight and the output are rounded to fp16, 2^-11 each; a score is exact in fp32 but for its last place, which
    the exponential multiplies by the score (up to 1e4 powers of two at 2^-24)."""
    from hqekv_amd.prompt_attention import prompt_attention
    g = torch.Generator(device=dev).manual_seed(T)
    q = torch.randn(B, Hq, T, 128, generator=g, device=dev, dtype=torch.float16) * 0.5
    k, v = (torch.randn(B, Hq // 4, T, 128, generator=g, device=dev, dtype=torch.float16) for _ in range(2))
    q[..., 0] = 16.0
    ramp = torch.arange(T, device=dev, dtype=torch.float64) * (climb / 32 * 0.6931471805599453 * 128 ** 0.5 / 16.0)
    k[..., 0] = (-ramp if down else ramp).clamp(-6e4, 6e4).half()
    out = prompt_attention(q, k, v, 128 ** -0.5)
    keep = torch.ones(T, T, dtype=torch.bool, device=dev).tril()
    for h in (0, Hq - 1):
        s = (q[-1, h].double() @ k[-1, h // 4].double().t().contiguous()) * 128 ** -0.5
        ref = s.masked_fill(~keep, float("-inf")).softmax(-1) @ v[-1, h // 4].double()
        got = out[-1, h] if out.shape[1] == Hq else out.transpose(1, 2)[-1, h]
        torch.testing.assert_close(got.double(), ref, rtol=3e-3, atol=3e-3)
