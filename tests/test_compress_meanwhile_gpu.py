"""What a compression lets its caller queue in the meantime (``cache_policy.compress(meanwhile=)``): called once on every
route -- prepared in C++, the gathers, the step engine -- and the cache that comes out is the same; what it raises is raised."""
import pytest
import torch

from hqekv_amd import cache_policy
from hqekv_amd.public_func import last_attn_weights, rank_blocks

pytestmark = pytest.mark.gpu


def _compress(dev, ranked_on_device, engine, meanwhile, ahead=lambda: None):
    g = torch.Generator().manual_seed(4)
    k, v = (torch.randn(1, 2, 330, 128, generator=g).half().to(dev) for _ in range(2))
    imp = torch.rand(320, generator=g).half().to(dev)
    lw = last_attn_weights(20)
    lw.set_max_length(400)
    lw.weights = torch.rand(20, 400, generator=g).half().to(dev)
    order = rank_blocks(32, 10, imp)
    counts = torch.tensor([64, 0, 96, 96, 32, 32], dtype=torch.int32)
    ahead()
    pkv = cache_policy.compress((None,) * 39 + (k, v, 330), 320, 0, order if ranked_on_device else order.tokens(), counts, counts.clone(),
                                imp, "uniform_group", last_weights=lw, n_targets=6, engine=engine, meanwhile=meanwhile)
    return pkv + (lw.weights,)


def test_called_once_on_every_route(dev):
    ref = _compress(dev, False, "steps", None)
    for ranked_on_device in (False, True):
        for engine in (None, "steps"):
            calls = []
            got = _compress(dev, ranked_on_device, engine, lambda: calls.append(1))
            assert len(calls) == 1
            for a, b in zip(got, ref):
                assert torch.equal(a, b) if torch.is_tensor(a) else a == b
            with pytest.raises(KeyError, match="theirs"):
                _compress(dev, ranked_on_device, engine, lambda: {}["theirs"])


def test_the_wait_is_for_the_ranking_alone(dev):
    """Some ten milliseconds of work queued ahead and ten times as much by the call: the compression comes back while that is
    still running, with the same cache."""
    a = torch.randn(8192, 8192, dtype=torch.float16, device=dev)
    b = torch.empty_like(a)
    ran, ref = torch.cuda.Event(), _compress(dev, True, None, None)

    def work(n):
        for _ in range(n):
            torch.mm(a, a, out=b)

    def meanwhile():
        work(100)
        ran.record()

    for _ in range(2):   # (the first one's allocations and library handles may wait for the device)
        got = _compress(dev, True, None, meanwhile, lambda: work(10))
        waited = ran.query()
        torch.cuda.synchronize()
        for x, y in zip(got, ref):
            assert torch.equal(x, y) if torch.is_tensor(x) else x == y
    assert not waited
