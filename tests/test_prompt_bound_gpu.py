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


def test_error_of_long_rows(dev):
    """No larger than with a rescale at each larger score and the sum taken before the weights are rounded to fp16: 2.5204e-4 (2-norm,
    relative, against 64 bits) for these rows."""
    from hqekv_amd.prompt_attention import prompt_attention
    T, e, r = 8192, 0.0, 0.0
    for seed in range(4):
        g = torch.Generator(device=dev).manual_seed(seed + T)
        q, k, v = (torch.randn(1, h, T, 128, generator=g, device=dev).half() for h in (32, 8, 8))
        out = prompt_attention(q, k, v, 128 ** -0.5)
        out = out if out.shape[1] == 32 else out.transpose(1, 2)
        rows, keys = torch.arange(seed, T, 8, device=dev), torch.arange(T, device=dev)
        for h in range(0, 32, 4):
            s = (q[0, h, rows].double() @ k[0, h // 4].double().t().contiguous()) * 128 ** -0.5
            want = s.masked_fill_(keys[None] > rows[:, None], float("-inf")).softmax(-1) @ v[0, h // 4].double()
            e += (out[0, h, rows].double() - want).square().sum().item()
            r += want.square().sum().item()
    assert (e / r) ** 0.5 <= 2.5204e-4
