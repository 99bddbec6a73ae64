"""Which form of the quantisers a call takes (csrc/quant_pack.hip), on both sides of their lines: K through the token-major
kernels -- token groups that fill a block in part, head sizes around 128 channels, appended into a window of longer planes --
against the rows kernel on the transposed tensor, and both against the oracle where that is quick.  Every bit counts."""
import pytest
import torch

from oracle import hqe_oracle as O

pytestmark = pytest.mark.gpu


def _window(B, H, D, n, bits, dev, at, room):
    pf, cap = 32 // bits, at + n + room
    code = torch.full((B, H, D, cap // pf), -1, dtype=torch.int32, device=dev)
    s, z = (torch.full((B, H, D, cap // 32), 7.0, dtype=torch.float16, device=dev) for _ in range(2))
    return (code, s, z), (code[..., at // pf:(at + n) // pf], s[..., at // 32:(at + n) // 32], z[..., at // 32:(at + n) // 32])


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("B,H,n,D", [
    (1, 2, 32, 128), (2, 1, 96, 64), (1, 1, 128, 128), (1, 3, 160, 128), (1, 2, 288, 96), (2, 1, 64, 256), (1, 1, 128, 160),
    (1, 64, 1024, 128), (1, 64, 992, 128), (1, 256, 512, 128), (3, 85, 512, 128), (1, 1024, 224, 64), (1, 1030, 160, 64)])
def test_both_ways_to_quantise_k(dev, B, H, n, D, bits):
    from hqekv_amd.pack_unpack import quantize_pack_into, uniform_group_quantize_pack_last_dim
    from hqekv_amd import _lib
    assert _lib.load().hqekv_selftest_form(2, n // 32, B * H, bits) == (n <= 128 or -(-n // 256) * B * H * max(bits, 2) >= 2048)
    g = torch.Generator(device=dev).manual_seed(n + D + bits)
    k = torch.randn(B, H, n, D, generator=g, device=dev, dtype=torch.float16)
    k[0, 0, :32] = 0.0
    k[0, 0, 5, ::3] = -0.0                     # a group of zeros of both signs
    k[-1, -1, -32:, 1] = 3.0                   # a constant group
    k[-1, -1, -1, 0] = float("inf")
    whole, into = _window(B, H, D, n, bits, dev, 64, 32)
    quantize_pack_into(k.transpose(2, 3), bits, *into)
    ref = uniform_group_quantize_pack_last_dim(k.transpose(2, 3).contiguous(), 32, bits)
    for got, want in zip(into, ref):
        assert torch.equal(got.contiguous().view(torch.int16 if got.dtype == torch.float16 else torch.int32),
                           want.view(torch.int16 if want.dtype == torch.float16 else torch.int32))
    for t, v in zip(whole, (-1, 7.0, 7.0)):    # nothing outside the window
        rest = t.clone()
        lo = 64 // 32 if t.dtype == torch.float16 else 64 * bits // 32
        m = n // 32 if t.dtype == torch.float16 else n * bits // 32
        rest[..., lo:lo + m] = v
        assert bool((rest == v).all())
    if B * H * n * D <= 1 << 16:
        for got, want in zip(ref, O.uniform_group_quantize_pack_last_dim(k.transpose(2, 3).contiguous().cpu(), 32, bits)):
            assert torch.equal(got.cpu().view(torch.int16 if got.dtype == torch.float16 else torch.int32),
                               want.view(torch.int16 if want.dtype == torch.float16 else torch.int32))


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("n", [131072 - 32, 131072, 131072 + 33])
def test_rows_in_parts_equal_the_whole(dev, n, bits):
    """Four groups per quad of lanes from 524288 groups on; fewer in halves of the same tensor."""
    from hqekv_amd.pack_unpack import uniform_group_quantize_pack_last_dim
    from hqekv_amd import _lib
    assert [_lib.load().hqekv_selftest_form(1, 4 * t, 0, 0) for t in (n, n // 2 + 1)] == [4 if n >= 131072 else 1, 1]
    v = torch.randn(1, 1, n, 128, generator=torch.Generator(device=dev).manual_seed(n), device=dev, dtype=torch.float16)
    whole = uniform_group_quantize_pack_last_dim(v, 32, bits)
    cut = n // 2 + 1
    parts = [uniform_group_quantize_pack_last_dim(x.contiguous(), 32, bits) for x in (v[:, :, :cut], v[:, :, cut:])]
    for w, a, b in zip(whole, *parts):
        assert torch.equal(w.view(torch.int16), torch.cat([a, b], 2).view(torch.int16))
