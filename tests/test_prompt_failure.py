"""A prompt whose attention fails (out of memory, say) leaves the layer's importance ring as it was, whatever the ring held and
wherever the attention is queued: at once, or behind the ranking of the prompt's compression."""
import pytest
import torch

from hqekv_amd import decode_layer

# (a prompt of 70 tokens has two blocks, which stay fp16; more are quantised, on the GPU alone)
PROMPTS = [("cpu", 7), ("cpu", 31), ("cpu", 70)] + [pytest.param("cuda", T, marks=pytest.mark.gpu) for T in (7, 31, 70, 330)]


def _prompt(T, device, seed):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(1, h, T, 128, generator=g).to(device, torch.float16) for h in (32, 8, 8))


def _ring(layer):
    lw = layer.last_weights
    return None if lw.weights is None else lw.weights.clone(), lw.kv_seq_len, lw.next_line


@pytest.mark.parametrize("device,T", PROMPTS)
@pytest.mark.parametrize("held", [0, 5, 40])
def test_ring_is_as_before(monkeypatch, device, T, held):
    layer = decode_layer.HqeAttentionLayer(128, bit_0=0.2, bit_4=0.5, bit_2=0.3)
    layer.set_max_length(400)
    if held:   # rows of an earlier prompt, no reset since
        layer(*_prompt(held, device, 1))
        layer.current_length = layer.history_reserve_length = 0
    before = _ring(layer)

    def fails(*_):
        raise torch.OutOfMemoryError("no room")

    with monkeypatch.context() as m:
        m.setattr(decode_layer, "gqa_prompt_attention", fails)
        with pytest.raises(torch.OutOfMemoryError):
            layer(*_prompt(T, device, 2))
    after = _ring(layer)
    assert after[1:] == before[1:] and (after[0] is None) == (before[0] is None)
    assert before[0] is None or torch.equal(after[0], before[0])
    # and the prompt that follows is what it would have been
    layer.current_length = 0
    out = layer(*_prompt(T, device, 2))[0]
    other = decode_layer.HqeAttentionLayer(128, bit_0=0.2, bit_4=0.5, bit_2=0.3)
    other.set_max_length(400)
    if held:
        other(*_prompt(held, device, 1))
        other.current_length = other.history_reserve_length = 0
    assert torch.equal(out, other(*_prompt(T, device, 2))[0])
    assert torch.equal(layer.last_weights.weights, other.last_weights.weights) and _ring(layer)[1:] == _ring(other)[1:]
