"""The few-rows projection kernel on its edges: partial row and column tiles,
partial K slices, weight rows split over two buffers off every tile, and each
tile choice (by row count), fp32 and bf16.

Bound: a projection is one fp32 sum of K products (exact for bf16 operands, one
rounding each for fp32) in partial sums, so an element is off from float64 by
at most (K + 8) 2^-24 sum |x w|.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _project(dev, M, r, K, bf16, of=None):
    """projections [M, 2r] of a window forward (one node per batch element) with its operands: the first M rows of
    `of` rows."""
    import jakal_net_native as jn

    of = of or M
    g = torch.Generator().manual_seed(of * 131 + r * 17 + K)
    X = torch.randn(of, 1, K, generator=g)[:M].to(dev, torch.bfloat16 if bf16 else torch.float32)
    U, V = (torch.randn(r, K, generator=g).to(dev) for _ in range(2))
    ps, w = torch.randn(M, 1, generator=g).to(dev), torch.ones(r, device=dev)
    ds, proj = torch.empty(M, 1, device=dev), torch.full((M, 2 * r), float("nan"), device=dev)
    dv, idx = torch.empty_like(X), torch.empty(M, 1, 1, device=dev, dtype=torch.int32)
    score = torch.empty(M, 1, 1, device=dev)
    fn = jn._LIB.jn_propagation_window_forward_bf16 if bf16 else jn._LIB.jn_propagation_window_forward
    p = jn._ptr
    jn._check(fn(p(X), p(ps), p(X), p(U), p(V), p(w), None, M, 1, K, K, r, 0, 0, p(ds), p(dv), p(proj), p(idx),
                 p(score), jn._stream(dev)))
    torch.cuda.synchronize()
    return X[:, 0].double(), U, V, proj


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M,r,K", [
    (1, 1, 8), (16, 8, 32), (17, 9, 40), (33, 32, 520), (1500, 33, 64), (1537, 64, 72), (3100, 24, 200),
    (4111, 64, 96), (8209, 64, 136), (8209, 20, 24), (16384, 64, 64), (16385, 64, 64), (32768, 16, 32),
    (40, 130, 264),
])
def test_projection_edges(M, r, K, bf16):
    dev = torch.device("cuda:0")
    X, U, V, proj = _project(dev, M, r, K, bf16)
    W = torch.cat([U, V])
    W = (W.bfloat16() if bf16 else W).double()
    want, scale = X @ W.t(), X.abs() @ W.abs().t()
    assert ((proj.double() - want).abs() <= (K + 8) * 2.0 ** -24 * scale).all()


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("Ns,Nd,r", [(100, 37, 24), (37, 300, 64), (520, 16, 8)])
def test_two_projections_in_one_launch(Ns, Nd, r, bf16):
    """A transition's source and destination projections, of unequal rows and widths, against torch."""
    import jakal_net as J

    dev, B, Ds, Dd = torch.device("cuda:0"), 3, 72, 136
    g = torch.Generator().manual_seed(Ns + Nd)
    route = J.LowRankBilinearRoute(Ds, Dd, rank=r).to(dev)
    dt = torch.bfloat16 if bf16 else torch.float32
    a, b = (torch.randn(B, n, d, generator=g).to(dev, dt) for n, d in ((Ns, Ds), (Nd, Dd)))
    val_proj = lambda v: v[..., :1].expand(*v.shape[:-1], Dd)  # noqa: E731
    op = J.SparseTransition(route, topk=Nd, val_proj_fn=val_proj, implementation="native")
    src = J.Layer(Ds, Ns, torch.randn(B, Ns, generator=g).to(dev, dt), a)
    dst = J.Layer(Dd, Nd, torch.zeros(B, Nd, device=dev, dtype=dt), b)
    with torch.no_grad():
        got = op.compute_delta(src, dst)
        if bf16:
            for p in (route.source_proj.weight, route.target_proj.weight):
                p.copy_(p.bfloat16())
        f = lambda layer: J.Layer(layer.dim, layer.num_nodes, layer.state.double(), layer.val.double())  # noqa: E731
        op.double().implementation = "reference"
        want = op.compute_delta(f(src), f(dst))
    tol = 2e-2 if bf16 else 1e-5
    assert (got.delta_val.double() - want.delta_val).norm() <= tol * want.delta_val.norm()


@pytest.mark.parametrize("M,r,bf16,rows", [
    (4096, 64, False, True), (4097, 64, False, False), (4080, 64, True, True), (4081, 64, True, False),
    (1024, 256, False, True), (1025, 256, False, False), (1008, 256, True, True), (1009, 256, True, False),
    (16384, 129, False, True), (16385, 129, False, False), (32768, 32, True, True), (32769, 32, True, False),
    (13632, 65, False, True), (13633, 65, False, False), (16384, 65, False, False), (16384, 65, True, True),
    (24576, 41, False, True), (24576, 57, False, False),  # three 64 x 64 tiles per CU, half and nearly filled
])
def test_rows_kernel_on_both_sides_of_its_line(M, r, bf16, rows):
    """Three-term and bf16 products of at most 2048 and fewer than 2048 tiles of 16 x 16, others by their rows, fp32
    ones but for those that fill three 64 x 64 tiles per CU."""
    import jakal_net_native as jn

    jn.profile_enable(True)
    try:
        _project(torch.device("cuda:0"), M, r, 64, bf16)
        names = [n for n in jn.profile_collect() if "project" in n]
    finally:
        jn.profile_enable(False)
    assert len(names) == 1 and names[0].startswith("gemm_rows_kernel") == rows, names


@pytest.mark.parametrize("r,K,bf16,of", [
    (64, 136, False, 4200),   # three-term: a call of one tile of rows more than the line, and of fewer
    (80, 520, False, 3300),
    (64, 136, True, 4200),    # bf16 MFMAs
    (96, 264, True, 2900),
    (40, 520, False, 32800),  # fp32 MFMAs, four chains
    (64, 72, False, 40),      # (too few rows for the MFMA tile kernels)
    (33, 136, True, 32800),   # the same on widened bf16 rows
])
def test_rows_kernel_has_the_bits_of_the_tile_kernel(r, K, bf16, of):
    """The rows of a large call, on the kernel that the rows kernel stands for, and the same rows in calls that it
    takes: top-k selections downstream must not depend on the number of rows."""
    import jakal_net_native as jn

    dev = torch.device("cuda:0")
    fp32_mfma = 2 * r < 128 or of < 128

    def run(M, forced=0):
        jn.set_gemm_tile(forced)
        jn.profile_enable(True)
        try:
            out = _project(dev, M, r, K, bf16, of)[3]
            names = [n for n in jn.profile_collect() if "project" in n]
        finally:
            jn.profile_enable(False)
            jn.set_gemm_tile(0)
        return out, names[0].startswith("gemm_rows_kernel")

    want, on_rows = run(of, 64 if fp32_mfma else 0)
    assert not on_rows
    for M in {1, 17, 40, 200, 1040, 2500, of - 1}:
        got, on_rows = run(min(M, of))
        if on_rows and (fp32_mfma or M >= 128):  # (below 128 rows every wide projection is one of fp32 MFMAs)
            assert torch.equal(got, want[:M]), M
        assert on_rows or M > 1040, M
