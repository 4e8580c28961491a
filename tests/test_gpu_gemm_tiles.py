"""Every GEMM workgroup tile (32 x 32, 64 x 64 and 128 x 128) and the automatic
choice (0: the fp32 projection GEMMs of 128+ extents on bf16 thirds) against
the oracle.

The library picks the tile per call from the output extents; these tests force
each tile in turn (jn_set_gemm_tile; 32 applies to the projection products and
their gradients, 64 to the others) on ops whose extents are ragged against
every tile, so every GEMM of the forward and backward passes (projections,
their input and weight gradients, dense scores, aggregation and its
gradients) runs partial tiles, unaligned rows and split-K under every tiling.
The 128 x 128 kernel has preconditions (extents and strides in float4 units,
B split at a multiple of 16); shapes that miss them run the 64 x 64 kernel
even when 128 is forced, and are included too.
Tolerances are those of the per-op tests (fp32: rtol 1e-4, atol 1e-5, or
for long sums within twice the error of an fp32 torch evaluation).
"""

import numpy as np
import pytest
import torch

import jakal_oracle as O
from parity import torch32_propagation
import test_gpu_bf16 as TB
import test_gpu_dense as TD
import test_gpu_topk as TT
import test_gpu_transition as TR
import test_gpu_window as TW

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[0, 32, 64, 128])
def tile(request):
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import jakal_net_native as jn

    jn.set_gemm_tile(request.param)
    yield request.param
    jn.set_gemm_tile(0)


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def test_dense_ragged(dev, tile):
    import jakal_net_native as jn

    B, N, D, r = 2, 200, 72, 12
    g, state, val, U, V, w = TD._inputs(4401, B, N, D, r)
    pv_cpu = torch.randn(B, N, D, generator=g)
    w_hat = w / w.norm()
    X = val.to(dev).requires_grad_(True)
    ps = state.to(dev).requires_grad_(True)
    pv = pv_cpu.to(dev).requires_grad_(True)
    Ud, Vd, wd = (t.to(dev).requires_grad_(True) for t in (U, V, w_hat))
    bd = torch.tensor(0.1, device=dev, requires_grad=True)
    ds, dv = jn.propagation_dense("low_rank_bilinear", wd, bd, Vd, None, Ud, None, "softsign", X, ps, pv, None, N, N)
    gds, gdv = torch.randn(B, N, generator=g), torch.randn(B, N, D, generator=g)
    torch.autograd.backward([ds, dv], [gds.to(dev), gdv.to(dev)])
    gr = O.propagation_backward(TD._np(val), TD._np(state), TD._np(pv_cpu), TD._np(U), TD._np(V), TD._np(w), 0.1,
                                TD._np(gds), TD._np(gdv), mode="dense", kind="softsign")
    t32 = torch32_propagation(dev, val, state, pv_cpu, U, V, w_hat, 0.1, np.ones((B, N, N), dtype=bool), "softsign",
                              gds, gdv)
    TD.compare_propagation(gr, t32, ds, dv, X, ps, pv, Ud, Vd, wd, bd)


def test_dense_small(dev, tile):
    TD.test_dense_forward_backward_matches_oracle(dev, "signed_abs_softmax", True, 37, False)


def test_dense_softsign_odd_columns(dev, tile):
    # 150 columns (not a multiple of 4): the softsign epilogue stores element-wise from the accumulators
    TD._check_dense(dev, "softsign", True, 150, True, B=2, D=24, r=6)


def test_topk_propagation(dev, tile):
    TT.test_propagation_topk_forward_backward_matches_oracle(dev, "softsign", True, 8)


def test_transition_odd(dev, tile):
    TR._run(dev, 3003, B=3, Ns=37, Nd=29, Dsrc=13, Ddst=7, r=3, topk=5, temperature=0.9, kind="signed_abs_softmax",
            with_bias=False)


@pytest.mark.parametrize("r", [40, 48])  # route weights split at r: 48 keeps the 128 x 128 kernel, 40 does not
def test_transition_medium(dev, tile, r):
    TR._run(dev, 3005, B=2, Ns=300, Nd=140, Dsrc=136, Ddst=72, r=r, topk=8, temperature=1.2, kind="softmax")


@pytest.mark.parametrize("compress", ["softsign", "signed_abs_softmax"])
def test_causal_dense(dev, tile, compress):
    # full causal windows run the dense products with causal K ranges and skip
    # the score tiles above the diagonal (softsign epilogue), under both tiles
    TW.test_full_causal_window_runs_dense(dev, compress, True, 0)


@pytest.mark.parametrize("mode", ["topk", "window"])
def test_bf16_layers(dev, tile, mode):
    # bf16 X in the projection (A), weight-gradient (B) and input-gradient (C)
    # GEMMs; rank 16 splits the weight operands at a multiple of 16, so the
    # 128 x 128 kernel takes all three uses when forced
    TB.run_bf16_propagation(dev, mode, B=2, N=160, D=40, r=16, k=8, seed=5003)


@pytest.mark.parametrize("D,r,separate_pv", [(136, 64, True), (512, 64, False), (200, 96, True)])
def test_fp32_projection_gemms_in_bf16_thirds(dev, D, r, separate_pv):
    """The automatic choice (tile 0) runs the fp32 projection, input-gradient
    and weight-gradient GEMMs with extents of 128 and more on gemm_x3_kernel
    (each fp32 operand split exactly into three bf16 terms, six bf16 MFMA
    products): ragged K (D = 136, 200) and N tails, the addend of grad X when
    pv is X, split-K over the rows; the fp32 tolerance of the per-op tests."""
    TT._run_topk(dev, TT._c1_inputs(seed=4500 + D, B=2, N=640, D=D, r=r), "softsign", separate_pv, 16,
                 min_checkable=0.5)


@pytest.mark.parametrize("B,N,D", [(1, 128, 128), (63, 132, 136), (64, 132, 136)])
def test_mfma_tiles_on_both_sides_of_the_line(dev, B, N, D):
    """The three-term GEMMs take 64 x 64 tiles below 256 tiles of 128 x 128: the
    smallest product (whole tiles), and ragged ones of 252 and 256 tiles."""
    TD._check_dense(dev, "softsign", True, N, True, B=B, D=D, r=16)


def test_bf16_product_is_the_same_on_both_tiles(dev):
    """The values of 64 dense bf16 transitions are summed on 256 tiles of 128 x
    128, those of 63 on 64 x 64 (the scores of both on the same kernel): every
    element keeps its chain over K, so the results are the same bit for bit."""
    import jakal_net_native as jn

    B, Ns, Nd, D, r = 64, 264, 136, 136, 16
    g = torch.Generator().manual_seed(4600)
    src, dst, pv = (torch.randn(B, n, D, generator=g).bfloat16().to(dev) for n in (Ns, Nd, Ns))
    ps = torch.randn(B, Ns, generator=g).bfloat16().to(dev)
    Ws, Wt = ((torch.randn(r, D, generator=g) / D**0.5).to(dev) for _ in range(2))
    w = (torch.rand(r, generator=g) + 0.5).to(dev)

    def run(n):
        rho = torch.nn.functional.softplus(ps[:n].float())
        return jn.transition_pairwise_dense("low_rank_bilinear_route", Ws, None, Wt, None, w, None, None, None, None,
                                            None, "softmax", 1.0, rho, src[:n], dst[:n], ps[:n], pv[:n], Ns, Nd)[1]

    assert torch.equal(run(64)[:63], run(63))


@pytest.mark.parametrize("compress,causal,separate_pv", [
    ("softsign", True, True), ("softsign", False, True), ("signed_abs_softmax", True, False),
    ("signed_entmax15", False, True),
])
def test_bf16_dense_products(dev, tile, compress, causal, separate_pv):
    # the bf16 dense products on 64- and 128-wide MFMA tiles: softsign epilogue, causal K ranges, ragged extents
    TB.test_bf16_dense_variants(dev, None, compress, causal, separate_pv, None)


@pytest.mark.parametrize("compress", ["softmax", "signed_abs_softmax"])
def test_bf16_route_products(dev, tile, compress):
    TB.test_bf16_dense_transition(dev, compress)


def _bf16_dense_step(dev, routes):
    """Outputs and gradients of a causal bf16 dense layer, and of a bf16 dense transition."""
    import jakal_net_native as jn

    B, N, Nd, D, r = 2, 264, 136, 200, 18
    g = torch.Generator().manual_seed(4700)
    leaf = lambda *s, dt=torch.float32: torch.randn(*s, generator=g).to(dev, dt).requires_grad_(True)  # noqa: E731
    X, dst = leaf(B, N, D, dt=torch.bfloat16), leaf(B, Nd, D, dt=torch.bfloat16)
    ps, w, U, V = leaf(B, N), leaf(r), leaf(r, D), leaf(r, D)
    out = jn.propagation_dense("low_rank_bilinear", w, None, V, None, U, None, "softsign", X, ps, X, None, N, N,
                               _causal=True)
    if routes:
        out += jn.transition_pairwise_dense("low_rank_bilinear_route", U, None, V, None, w, None, None, None, None,
                                            None, "softmax", 1.0, torch.nn.functional.softplus(ps), X, dst, ps, X, N,
                                            Nd)
    gs = [torch.randn(o.shape, generator=g).to(dev, o.dtype) for o in out]
    return [*out, *torch.autograd.grad(out, [X, ps, w, U, V], gs)]


@pytest.mark.parametrize("forced", [64, 128])
def test_forced_tile_reaches_the_mfma_products(dev, forced):
    """The bf16 MFMA kernels of the dense products run on the forced tile (their last template argument), whatever
    the grid."""
    import jakal_net_native as jn
    from torch.profiler import ProfilerActivity, profile

    try:
        jn.set_gemm_tile(forced)
        _bf16_dense_step(dev, True)
        with profile(activities=[ProfilerActivity.CUDA]) as prof:
            _bf16_dense_step(dev, True)
            torch.cuda.synchronize()
    finally:
        jn.set_gemm_tile(0)
    names = [e.key for e in prof.key_averages() if "gemm_bf16_kernel<" in e.key]
    assert len(names) >= 6 and all(f", {forced}>" in n for n in names), names


def test_bf16_dense_step_is_the_same_on_both_tiles(dev):
    """Every element of the MFMA products keeps its chain over K on either tile, so everything but the weight
    gradients, fp32 products that a forced tile moves as well, is the same bit for bit.  (Rank 18 keeps the other fp32
    products on their 64 x 64 tiles.)"""
    import jakal_net_native as jn

    results = []
    try:
        for forced in (64, 128):
            jn.set_gemm_tile(forced)
            results.append(_bf16_dense_step(dev, False))
    finally:
        jn.set_gemm_tile(0)
    for i, (a, b) in enumerate(zip(*results)):
        if i < len(results[0]) - 2:
            assert torch.equal(a, b), i
        else:
            assert (a - b).norm() <= 1e-5 * b.norm()


def test_three_term_products_are_the_same_on_both_tiles(dev):
    """A window layer's projections and input gradient on 256 tiles of 128 x 128 and on 255, which take 64 x 64: every
    element keeps its chain over K, so the rows both calls have are the same bit for bit."""
    import jakal_net_native as jn

    B, N, D, r = 256, 128, 128, 64
    g = torch.Generator().manual_seed(4800)
    val, state, gs, gv = (torch.randn(B, N, *s, generator=g).to(dev) for s in ((D,), (), (), (D,)))
    U, V = ((torch.randn(r, D, generator=g) / D**0.5).to(dev) for _ in range(2))
    w = torch.full((r,), r**-0.5, device=dev)

    def run(n):
        X, ps = val[:n].clone().requires_grad_(True), state[:n].clone().requires_grad_(True)
        out = jn.propagation_window("low_rank_bilinear", w, None, V, None, U, None, "softsign", X, ps, X, 16, N, N)
        return [t[:B - 1] for t in (*out, *torch.autograd.grad(out, [X, ps], [gs[:n], gv[:n]]))]

    for a, b in zip(run(B), run(B - 1)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rows,D,tile", [(20480, 256, 128), (16384, 256, 64), (20480, 128, 64)])
def test_weight_gradient_tile_beside_the_input_gradient(dev, rows, D, tile):
    """The fp32 weight gradient takes 128-wide tiles beside the input gradient (on the second stream) of more than
    16,384 rows where they make 128 workgroups, 64-wide ones by itself, and the same bits either way."""
    import jakal_net_native as jn
    from torch.profiler import ProfilerActivity, profile

    g = torch.Generator().manual_seed(rows + D)
    N, r = 2048, 64
    X, ps = (torch.randn(*s, generator=g).to(dev).requires_grad_(True) for s in ((rows // N, N, D), (rows // N, N)))
    U, V = (torch.randn(r, D, generator=g).to(dev).requires_grad_(True) for _ in range(2))
    w, gv = torch.ones(r, device=dev), torch.randn(rows // N, N, D, generator=g).to(dev)

    def step():
        out = jn.propagation_window("low_rank_bilinear", w, None, V, None, U, None, "softsign", X, ps, X, 31, N, N)
        return torch.autograd.grad(out[1], [X, U, V], gv)

    grads = []
    try:
        for side, want in ((True, tile), (False, 64)):
            jn.set_side_streams(side)
            step()
            with profile(activities=[ProfilerActivity.CUDA]) as prof:
                grads.append(step())
                torch.cuda.synchronize()
            names = [e.key for e in prof.key_averages() if "gemm_x3_kernel<false, false, 2," in e.key]
            assert len(names) == 1 and all(f", {want}>" in n for n in names), names
    finally:
        jn.set_side_streams(True)
    assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("bf16,B,aggregate,value_grad", [
    (False, 16, 64, 64), (False, 17, 64, 128), (False, 24, 64, 128), (False, 25, 128, 128),  # 8 wide tiles each
    (True, 24, 64, 64), (True, 25, 64, 128), (True, 31, 64, 128), (True, 32, 128, 128),
])
def test_tile_of_a_dense_product(dev, bf16, B, aggregate, value_grad):
    """Which tile the N x N products of a layer take on either side of their lines, by use."""
    import re

    import jakal_net_native as jn
    from torch.profiler import ProfilerActivity, profile

    N, D, r = 1024, 128, 8
    dt = torch.bfloat16 if bf16 else torch.float32
    X = torch.randn(B, N, D, device=dev).to(dt).requires_grad_(True)
    ps, w = torch.randn(B, N, device=dev), torch.ones(r, device=dev)
    U, V = (torch.randn(r, D, device=dev) for _ in range(2))

    def step():
        out = jn.propagation_dense("low_rank_bilinear", w, None, V, None, U, None, "signed_abs_softmax", X, ps, X, None,
                                   N, N)
        out[1].backward(torch.ones_like(out[1]))
        torch.cuda.synchronize()

    step()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        step()
    tile = {}
    for e in prof.key_averages():
        m = re.search(r"gemm_(x3|bf16)_kernel<(.*?)>", e.key)
        if m:
            *_, use, t = m.group(2).split(",")
            tile[int(use)] = int(t)
    uses = (19, 20) if bf16 else (4, 6)
    assert tuple(tile[u] for u in uses) == (aggregate, value_grad), tile


@pytest.mark.parametrize("B,tile", [(32, 64), (33, 128)])
def test_weight_gradient_tile_of_a_transition(dev, B, tile):
    """A transition's weight gradients, of two sides on two streams, from 32,768 rows on; the same bits on one stream."""
    import jakal_net_native as jn
    from torch.profiler import ProfilerActivity, profile

    g = torch.Generator().manual_seed(B)
    N, D, r = 1024, 256, 128
    rand = lambda *s: torch.randn(*s, generator=g).to(dev)  # noqa: E731
    src, dst, rho, ps = rand(B, N, D), rand(B, N, D), rand(B, N), rand(B, N)
    U, V = (rand(r, D).requires_grad_(True) for _ in range(2))
    w, gv = torch.ones(r, device=dev) / r, rand(B, N, D)

    def step():
        out = jn.transition_pairwise_topk("low_rank_bilinear_route", U, None, V, None, w, None, None, None, None, None,
                                          1.0, rho, src, dst, ps, src, 8, N, N)
        return torch.autograd.grad(out[1], [U, V], gv)

    grads = []
    try:
        for side, want in ((True, tile), (False, 64)):
            jn.set_side_streams(side)
            step()
            with profile(activities=[ProfilerActivity.CUDA]) as prof:
                grads.append(step())
                torch.cuda.synchronize()
            names = [e.key for e in prof.key_averages() if "gemm_x3_kernel<false, false, 2," in e.key]
            assert len(names) == 1 and f", {want}>" in names[0], names
    finally:
        jn.set_side_streams(True)
    assert all(torch.equal(a, b) for a, b in zip(*grads))
