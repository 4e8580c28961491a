"""Work is forked onto the second stream only where there is some: the grouping of small edge lists has no half that
could run beside the row pass, so calls on them wait for no event."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _waits(call):
    """hipStreamWaitEvent calls of one call (after one that creates streams and events)."""
    from torch.profiler import ProfilerActivity, profile

    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    counts = {e.key: e.count for e in prof.key_averages()}
    assert any(k.startswith("hip") and "Launch" in k for k in counts), "the profiler records no runtime calls"
    return sum(n for k, n in counts.items() if "StreamWaitEvent" in k)


@pytest.mark.parametrize("B,Ns,k,waits", [(16, 1024, 16, 0), (8, 2048, 16, 2)])
def test_transition_forward(B, Ns, k, waits):
    """2^18 routes: 16,384 of an element are grouped in one launch, 32,768 in a layout beside the coefficients."""
    import jakal_net as J

    dev, D, Nd = torch.device("cuda:0"), 64, 200
    g = torch.Generator().manual_seed(Ns)
    op = J.SparseTransition(J.LowRankBilinearRoute(D, D, rank=8), topk=k, implementation="native").to(dev)
    layer = lambda n: J.Layer(D, n, torch.randn(B, n, generator=g).to(dev),  # noqa: E731
                              torch.randn(B, n, D, generator=g).to(dev))
    src, dst = layer(Ns), layer(Nd)
    with torch.no_grad():
        assert _waits(lambda: op.compute_delta(src, dst)) == waits
