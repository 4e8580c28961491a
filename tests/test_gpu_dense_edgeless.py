"""bf16 dense softsign layers without an edge matrix, on the edges of their tiles:
partial 128-row and 64- and 32-column tiles, every value width (128 to 512),
ranks of one and two 32-wide planes and odd ones, both causal orders, batches in
one and in several launches, and a second backward of one forward.

The reference is float64 on the operands the layer has: bf16 values, weights
rounded to bf16, edges rounded to bf16 where they multiply values.  Tolerances,
as relative 2-norms: bf16 outputs 2^-8 (one rounding of the result and one of
the edges); fp32 state sums and score-scale gradients 2e-6 and 1e-5 (fp32
projections of K = D terms, fp32 products, sums over N); weight gradients
2^-8 (the projection gradient is rounded to bf16); the bias gradient, a sum of
N^2 terms of either sign, 2^-20 of the sum of their magnitudes.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _case(B, N, D, r, causal, separate, bias, seed):
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g).to(DEV)  # noqa: E731
    t = dict(X=rand(B, N, D).bfloat16(), ps=rand(B, N), U=rand(r, D) / D ** 0.5, V=rand(r, D) / D ** 0.5,
             w=1 + 0.2 * rand(r), b=rand(1)[0] if bias else None,
             pv=rand(B, N, D).bfloat16() if separate else None, gs=rand(B, N), gv=rand(B, N, D).bfloat16())
    return {k: v.requires_grad_(k not in ("gs", "gv")) if v is not None else None for k, v in t.items()}


def _run(t, causal):
    import jakal_net_native as jn

    pv = t["X"] if t["pv"] is None else t["pv"]
    N = t["X"].shape[1]
    return jn.propagation_dense("low_rank_bilinear", t["w"], t["b"], t["V"], None, t["U"], None, "softsign", t["X"],
                                t["ps"], pv, None, N, N, _causal=causal)


class _Round(torch.autograd.Function):
    """x rounded to bf16, the gradient of x itself."""

    @staticmethod
    def forward(ctx, x):
        return x.bfloat16().double()

    @staticmethod
    def backward(ctx, g):
        return g


def _reference(t, causal):
    d = {k: None if v is None else v.detach().double().requires_grad_(v.requires_grad) for k, v in t.items()}
    q, k = d["X"] @ _Round.apply(d["U"]).t() * d["w"], d["X"] @ _Round.apply(d["V"]).t()
    s = q @ k.transpose(1, 2) + (d["b"] if d["b"] is not None else 0)
    s.retain_grad()
    e = torch.nn.functional.softsign(s)
    if causal:
        e = e.tril()
    pv = d["X"] if d["pv"] is None else d["pv"]
    ds, dv = (e @ d["ps"].unsqueeze(-1)).squeeze(-1), _Round.apply(e) @ pv
    torch.autograd.backward([ds, dv], [d["gs"], d["gv"]])
    return ds, dv, d, s.grad


def _off(got, want, tol, what):
    err = float((got.detach().double() - want).norm() / want.norm())
    assert err <= tol, f"{what}: {err:.2e} > {tol:.0e}"


@pytest.mark.parametrize("B,N,D,r,causal,separate,bias", [
    (2, 712, 128, 1, False, False, True),
    (2, 768, 256, 32, False, True, False),
    (1, 1000, 384, 33, True, False, True),
    (2, 904, 512, 64, True, True, True),
    (3, 1032, 512, 20, False, False, True),
    (1, 776, 384, 64, False, True, False),
    (2, 1024, 128, 63, True, True, False),
])
@pytest.mark.parametrize("per_launch", [None, 1])
def test_edgeless_dense(B, N, D, r, causal, separate, bias, per_launch):
    import jakal_net_native as jn

    assert jn._LIB.jn_propagation_dense_edgeless_bf16(N, D, r, 0) == 1
    t = _case(B, N, D, r, causal, separate, bias, seed=N + D + r)
    if per_launch:
        jn.set_dense_edge_bytes(per_launch * N * N * 4)
    try:
        ds, dv = _run(t, causal)
        torch.autograd.backward([ds, dv], [t["gs"], t["gv"]], retain_graph=True)
        first = {k: v.grad.clone() for k, v in t.items() if v is not None and v.requires_grad}
        for v in t.values():
            if v is not None:
                v.grad = None
        torch.autograd.backward([ds, dv], [t["gs"], t["gv"]])
    finally:
        jn.set_dense_edge_bytes()
    wds, wdv, d, sg = _reference(t, causal)
    for k, v in first.items():
        assert torch.equal(v, t[k].grad), f"second backward: {k}"
    _off(ds, wds.detach(), 2e-6, "delta_state")
    _off(dv, wdv.detach(), 2 ** -8, "delta_val")
    _off(first["ps"], d["ps"].grad, 2e-6, "grad state")
    _off(first["X"], d["X"].grad, 2 ** -8, "grad values")
    for k in ("U", "V"):
        _off(first[k], d[k].grad, 2 ** -8, k)
    _off(first["w"], d["w"].grad, 1e-5, "w")
    if separate:
        _off(first["pv"], d["pv"].grad, 2 ** -8, "pv")
    if bias:
        assert abs(float(first["b"]) - float(d["b"].grad)) <= 2 ** -20 * float(sg.abs().sum())


def test_edgeless_rule():
    import jakal_net_native as jn

    ok = jn._LIB.jn_propagation_dense_edgeless_bf16
    assert ok(4096, 512, 64, 0) == 1
    for args in ((4096, 520, 64, 0), (4096, 640, 64, 0), (4096, 512, 65, 0), (4096, 512, 64, 1), (256, 512, 64, 0)):
        assert ok(*args) == 0


def _library_step(B, N, D, r, causal, edges):
    """Every output of one layer through the C entry points: over a kept edge matrix, or on scratch of its size."""
    import jakal_net_native as jn

    t = {k: v.detach() for k, v in _case(B, N, D, r, causal, True, True, seed=B + N + r).items()}
    L, p, st = jn._LIB, jn._ptr, jn._stream(DEV)
    ds, dv, proj = torch.empty(B, N, device=DEV), torch.empty_like(t["X"]), torch.empty(B * N, 2 * r, device=DEV)
    E = torch.empty(B * N * N * 4 + 256, device=DEV, dtype=torch.uint8)
    args = [p(t[k]) for k in ("X", "ps", "pv", "U", "V", "w", "b")]
    sizes = [B, N, D, D, r, 0, causal]
    out = [p(ds), p(dv), p(proj), p(E)]
    if edges:
        jn._check(L.jn_propagation_dense_forward_bf16(*args, *sizes, *out, st))
        ws_bytes = L.jn_propagation_dense_workspace_bytes(B, N, D, D, r, 0, 1)
    else:
        jn._check(L.jn_propagation_dense_forward_chunked_bf16(*args, *sizes, B, *out, E.numel(), st))
        ws_bytes = L.jn_propagation_dense_chunked_workspace_bytes(B, N, D, D, r, 0, B, 1)
    ws = torch.empty(ws_bytes, device=DEV, dtype=torch.uint8)
    grads = [torch.empty_like(t[k]) for k in ("X", "ps", "pv", "U", "V", "w", "b")]
    back = [p(proj), p(E), p(t["gs"]), p(t["gv"]), *sizes, 0]
    tail = [*map(p, grads), p(ws), ws_bytes, st]
    if edges:
        jn._check(L.jn_propagation_dense_backward_bf16(*args[:6], *back, 1, *tail))
    else:
        jn._check(L.jn_propagation_dense_backward_chunked_bf16(*args, *back, B, 0, *tail))
    torch.cuda.synchronize()
    return dict(zip(("delta_state", "delta_val", "X", "ps", "pv", "U", "V", "w", "b"), (ds, dv, *grads)))


@pytest.mark.parametrize("B,N,D,r,causal", [
    (37, 776, 128, 20, 0), (24, 1032, 256, 64, 1), (28, 904, 384, 48, 1), (26, 1000, 512, 32, 0), (24, 1024, 512, 64, 0),
])
def test_same_bits_as_over_an_edge_matrix(B, N, D, r, causal):
    """Rebuilding the edges keeps every product and every sum of the GEMMs over a stored edge matrix."""
    got, want = (_library_step(B, N, D, r, causal, edges) for edges in (False, True))
    for k in want:
        assert torch.equal(got[k], want[k]), k


@pytest.mark.parametrize("B,N,D,r", [(4, 520, 512, 33), (8, 256, 256, 17)])
def test_second_backward_where_one_matrix_is_too_small(B, N, D, r):
    """Layers whose operand layouts exceed one edge matrix but not the batch's: their edges are kept, and a second
    backward rebuilds them as the forward did."""
    import jakal_net_native as jn

    assert jn._LIB.jn_propagation_dense_edgeless_bf16(N, D, r, 0) == 0
    t = _case(B, N, D, r, False, True, True, seed=N)
    ds, dv = _run(t, False)
    grads = []
    for keep in (True, False):
        torch.autograd.backward([ds, dv], [t["gs"], t["gv"]], retain_graph=keep)
        grads.append({k: v.grad for k, v in t.items() if v.requires_grad})
        for v in t.values():
            v.grad = None
    for k in grads[0]:
        assert torch.equal(grads[0][k], grads[1][k]), k


@pytest.mark.parametrize("B,N,D,r,causal,separate,bias,per_launch", [
    (43, 712, 128, 1, False, False, True, None),
    (28, 776, 256, 32, False, True, False, None),
    (24, 1000, 384, 33, True, False, True, None),
    (24, 904, 512, 64, True, True, True, None),
    (22, 1032, 512, 20, False, False, True, None),
    (28, 776, 384, 64, False, True, False, None),
    (32, 1024, 128, 63, True, True, False, None),
    (63, 1024, 128, 40, False, True, True, 10),  # launches of 32 and 31
    (49, 1016, 512, 64, True, False, True, 16),  # 25 and 24
])
def test_edgeless_dense_on_full_grids(B, N, D, r, causal, separate, bias, per_launch):
    """The same at the batches from which the layer runs without an edge matrix."""
    import jakal_net_native as jn

    assert jn._LIB.jn_propagation_dense_edgeless_chunk_bf16(B, N, D, r, 0, int(causal), per_launch or B) > 0
    test_edgeless_dense(B, N, D, r, causal, separate, bias, per_launch)


@pytest.mark.parametrize("B,N,D,r,causal,edgeless", [
    (31, 704, 512, 64, False, False), (32, 704, 512, 64, True, True), (63, 512, 128, 8, False, False),
    (64, 512, 128, 8, True, True), (5, 3000, 512, 64, False, False), (6, 3000, 512, 64, False, True),
    (1, 4096, 512, 64, False, False), (4, 4096, 512, 64, False, True), (5, 4096, 512, 64, True, False),
    (6, 4096, 128, 64, True, True),
])
def test_kernels_of_a_batch(B, N, D, r, causal, edgeless):
    """Which kernels a layer runs on either side of the line (small grids leave most of the chip idle without edges)."""
    import jakal_net_native as jn

    t = _case(B, N, D, r, causal, False, True, seed=5)
    jn.profile_enable(True)
    try:
        ds, dv = _run(t, causal)
        torch.autograd.backward([ds, dv], [t["gs"], t["gv"]])
        torch.cuda.synchronize()
        names = "".join(jn.profile_collect())
    finally:
        jn.profile_enable(False)
    assert ("dense_score_grad_kernel" in names) == ("dense_aggregate_kernel<forward>" in names) == edgeless
    assert ("gemm_bf16_kernel<dense_edge_grad_bf16>" in names) != edgeless


def test_edgeless_forward_keeps_no_scratch():
    """Between forward and backward the layer holds its outputs and projections, not an edge matrix's worth of scratch."""
    B, N, D, r = 24, 1024, 512, 64
    t = _case(B, N, D, r, False, True, True, seed=9)
    _run(t, False)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated(DEV)
    ds, dv = _run(t, False)
    held = torch.cuda.memory_allocated(DEV) - before
    assert held <= B * N * (4 + 2 * D + 8 * r) + (1 << 20)
    torch.autograd.backward([ds, dv], [t["gs"], t["gv"]])
