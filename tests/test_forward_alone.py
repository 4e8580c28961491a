"""Calls that nothing records (no gradient wanted, no transform active) run an
op's forward by itself: same results as through its autograd function, for any
batch shape, stride and type, and the same errors."""

import pytest
import torch
from torch.autograd import forward_ad


def test_what_goes_through_the_autograd_function():
    import jakal_net_native as jn

    x, p = torch.zeros(2), torch.zeros(2, requires_grad=True)
    assert jn._records(x, p) and not jn._records(x, None)
    with torch.no_grad():
        assert not jn._records(x, p)
        with forward_ad.dual_level():
            assert jn._records(x)
        torch.func.vmap(lambda t: t if jn._records(t) else 1 / 0)(x)
        torch.jit.trace(lambda t: t + 0 if jn._records(t) else 1 / 0, (x,), check_trace=False)


def _ops(kind, dtype, dev, g):
    import jakal_net as J

    D, r = 40, 8
    if kind in ("topk_routes", "dense_routes"):
        route = J.LowRankBilinearRoute(D, D, rank=r)
        op = J.SparseTransition(route, topk=6, implementation="native") if kind == "topk_routes" else J.Transition(
            route, implementation="native")
        sizes = (19, 33)
    else:
        pair = J.LowRankBilinearPairwise(D, r)
        if kind == "heads":
            pair = J.MultiHeadPairwise([J.LowRankBilinearPairwise(D, r) for _ in range(2)])
        how = dict(sparse_type="window", window=7) if kind == "window" else dict(sparse_type="topk", topk=5)
        op = J.Propagation(pair, implementation="native") if kind == "dense" else J.SparsePropagation(
            pair, implementation="native", **how)
        sizes = (37,)
    return op.to(dev), sizes, D


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [(), (3,), (2, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["topk", "heads", "window", "dense", "topk_routes", "dense_routes"])
def test_forward_alone_equals_recorded(kind, dtype, batch):
    import jakal_net as J

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(5)
    torch.manual_seed(5)
    op, sizes, D = _ops(kind, dtype, dev, g)
    layers = []
    for n in sizes:
        val = torch.randn(*batch, D, n, generator=g).to(dev, dtype).transpose(-1, -2)  # strided rows
        state = torch.randn(*batch, n, 2, generator=g).to(dev, dtype)[..., 0]
        layers.append(J.Layer(dim=D, num_nodes=n, state=state, val=val))
    recorded = op.compute_delta(*layers)
    assert recorded.delta_val.requires_grad
    with torch.no_grad():
        alone = op.compute_delta(*layers)
    assert not alone.delta_val.requires_grad
    for a, b in ((recorded.delta_state, alone.delta_state), (recorded.delta_val, alone.delta_val)):
        assert a.dtype == b.dtype == dtype and torch.equal(a, b)


@pytest.mark.gpu
def test_mismatched_rows_and_forward_mode_still_raise():
    import jakal_net_native as jn

    dev = torch.device("cuda:0")
    X = torch.randn(2, 20, 8, device=dev)
    U, V, w = torch.randn(4, 8, device=dev), torch.randn(4, 8, device=dev), torch.ones(4, device=dev)
    call = lambda x, ps: jn.propagation_topk("low_rank_bilinear", w, None, V, None, U, None, "softsign", x, ps,  # noqa: E731
                                             x, 3, 8, 8)
    with pytest.raises(RuntimeError):
        call(X, torch.randn(2, 19, device=dev))
    with torch.no_grad(), forward_ad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        call(forward_ad.make_dual(X, X), torch.randn(2, 20, device=dev))
