"""Branches of the launch rules at the sizes where they can go wrong, against
the FP64 oracle: boundary fills whose two faces share a launch or run in turn,
the marches' segment counts on blocks too small to fill the chip, the x-line
kernels' segments, and the surrogate fallback's second pass over the cells of many Newton iterations."""
import os

import numpy as np
import pytest
import torch

from helpers import rel_err, to_np, to_torch

pytestmark = pytest.mark.gpu


def _state(shape, m, seed=3):
    import flame3d_amd.cases as cases
    grid = cases.skewed_grid(*shape)
    Q, rhoi = cases.random_state(grid, m, seed=seed, shock=True)
    return grid, Q, rhoi


@pytest.mark.parametrize("mech", ["air5", "h2_lidryer"])
@pytest.mark.parametrize("kinds", [(1, 2, 2, 1, 1, 3), (3, 1, 1, 3, 2, 3), (2, 1, 0, 1, 3, 3),
                                   (1, 1, 2, 2, 0, 0)])
def test_fill_pairs_of_faces(mech, kinds):
    """Every pairing of fill kinds on the smallest block (N = 4, where copy
    sources and periodic sources are nearest the nodes the other face
    writes); copies of values: equal bit for bit."""
    import flame3d_amd.abi as abi
    import flame3d_amd.mech as mm
    from oracle import Oracle
    m = mm.load(mech)
    shape = (4, 5, 4)
    grid, Q, rhoi = _state(shape, m)
    orc, ctx = Oracle(*shape, m), abi.Context(*shape, m, "fp64")
    inQ = [1.2, 300.0, 1.0, -2.0, 1.0e5, 310.0, 2.0e5]
    inr = list(np.linspace(0.1, 0.2, m.Ns))
    Qo, ro = to_np(Q), to_np(rhoi)
    Uo = orc.prim2c(Qo)
    Qg, rg, Ug = Q.cuda(), rhoi.cuda(), to_torch(Uo)
    orc.fill(kinds, Qo, Uo, ro, inQ, inr)
    ctx.set_boundary(kinds, inQ, inr)
    ctx.fill(Qg, Ug, rg)
    torch.cuda.synchronize()
    for got, ref in ((Qg, Qo), (Ug, Uo), (rg, ro)):
        assert np.array_equal(to_np(got), ref)
    ctx.close()


@pytest.mark.parametrize("shape", [(4, 4, 4), (65, 7, 5), (9, 33, 34), (70, 66, 9), (128, 4, 5),
                                   (257, 5, 4), (5, 127, 4), (66, 131, 70)])
@pytest.mark.parametrize("mech", ["air5", "h2_lidryer"])
def test_stage_on_small_and_ragged_blocks(mech, shape):
    """One FP64 stage on blocks of one short segment, several, a remainder
    segment and a partial wave (marches), and of x lines that take one to four
    waves or two segments of the fused x sweep: 1e-12 normwise per field, the
    FP64 path's parity bar."""
    import flame3d_amd.abi as abi
    import flame3d_amd.cases as cases
    import flame3d_amd.mech as mm
    from oracle import Oracle
    m = mm.load(mech)
    grid, Q, rhoi = _state(shape, m, seed=8)
    dt = cases.cfl_dt(grid, Q, 0.3)
    kinds = (2, 2, 2, 2, 1, 1)
    orc = Oracle(*shape, m)
    Qo, ro = to_np(Q), to_np(rhoi)
    U = orc.prim2c(Qo)
    M, J = [to_np(x) for x in grid.metrics], to_np(grid.J)
    ctx = abi.Context(*shape, m, "fp64")
    ctx.set_metrics([x.cuda() for x in grid.metrics], grid.J.cuda())
    ctx.set_boundary(kinds)
    Qg, rg, Ug = Q.cuda(), rhoi.cuda(), to_torch(U)
    orc.rk3_stage(1, U, orc.zeros(5), ro, orc.zeros(m.Ns), Qo, orc.workspace(), M, J, dt, kinds)
    ctx.rk3_stage(1, Ug, ctx.zeros(5), rg, ctx.zeros(m.Ns), Qg, dt)
    torch.cuda.synchronize()
    for got, ref in ((Qg, Qo), (Ug, U), (rg, ro)):
        assert rel_err(to_np(got), ref) < 1e-12
    ctx.close()


@pytest.mark.parametrize("maxiter", [1, 5, 6, 50])
@pytest.mark.parametrize("mech,shape", [("h2_lidryer", (32, 31, 9)), ("h2_lidryer", (5, 4, 4)),
                                        ("air5", (17, 9, 6))])
def test_fallback_equals_newton(mech, shape, maxiter):
    """Cells that the surrogate rejects (every reacting one: a chain bound of
    1e-30) are advanced by a pass over the list and those of more than five
    iterations, or of a failed first step, by the half-wave solve.  Both form
    every sum in the order of the Newton mode: equal bit for bit, also where
    no substep count converges and the cell stays unreacted, and (one
    iteration allowed) where more cells are slow than the second pass takes."""
    import flame3d_amd.abi as abi
    import flame3d_amd.cases as cases
    import flame3d_amd.mech as mm
    import flame3d_amd.surrogate as sur
    m = mm.load(mech)
    h2 = mech == "h2_lidryer"
    if h2:
        Q, r = cases.chem_cells(shape, m, seed=7)
        dt = sur.DT
    else:
        Q, r = cases.chem_cells_air(shape, m, seed=7, T_range=(1500.0, 6000.0),
                                    P_atm=(0.02, 0.1))
        dt = sur.AIR_DT
    Q, r = Q.cuda().contiguous(), r.cuda().contiguous()
    U = torch.zeros((5,) + tuple(Q.shape[1:]), dtype=torch.float64, device="cuda")
    ctx = abi.Context(*shape, m, "fp64")
    path = os.path.join(os.path.dirname(sur.DEFAULT_PATH), "air5_surrogate.npz")
    sur.attach(ctx, *([] if h2 else [path]), chain_max=1e-30)
    Un, Qn, rn = U.clone(), Q.clone(), r.clone()
    it = torch.zeros(shape[::-1], dtype=torch.int32, device="cuda")
    ctx.chem_newton(Un, Qn, rn, dt, maxiter, 1e-10, 1e-6, iters=it)
    st = torch.zeros(shape[::-1], dtype=torch.int8, device="cuda")
    nfb = int(ctx.nn_chem(U, Q, r, dt, maxiter, 1e-10, 1e-6, status=st))
    torch.cuda.synchronize()
    print(f"\n[fallback] {mech} {shape} maxiter {maxiter}: {nfb} of {st.numel()} rejected, "
          f"iterations up to {int(it.abs().max())}, {int((it < 0).sum())} left unreacted")
    back = st != 1
    assert int(back.sum()) > st.numel() // 2
    if h2 and st.numel() > 1000:
        assert bool((back & ((it.abs() > 5) | (it < 0))).any())  # the second pass had work
    for got, ref in ((U, Un), (Q, Qn), (r, rn)):
        assert torch.equal(sur.interior(got)[back.flatten()], sur.interior(ref)[back.flatten()])
    ctx.close()


@pytest.mark.parametrize("mech,nx,scheme", [
    ("air5", 4, None), ("air5", 56, "weno7"), ("air5", 60, None), ("h2_lidryer", 61, None),
    ("h2_lidryer", 128, "weno7"), ("air5", 129, None), ("h2_lidryer", 129, None),
    ("h2_lidryer", 256, None), ("h2_lidryer", 257, "weno7"), ("air5", 304, "weno7"),
    ("air5", 305, None), ("h2_lidryer", 305, None), ("air5", 609, "weno7")])
def test_x_line_segments(mech, nx, scheme):
    """The fused FP32 stage on x lines at the edges of its rules: the smallest,
    those whose cells and staged points just fill or just exceed a number of
    waves, the largest and one more of each LDS tile, and lines of two and three
    segments; the granular stage's bars of test_gpu_sweeps."""
    import flame3d_amd.abi as abi
    from test_gpu_sweeps import _cmp, _stage_pair
    sc = {"recon_kind": abi.RECON_WENO7} if scheme else None
    print(f"\n[x lines] {mech} nx={nx} {scheme}", flush=True)
    f, g = _stage_pair(mech, (nx, 5, 6), scheme=sc)
    _cmp(f[0], g[0], "dU", 1e-4)
    _cmp(f[1], g[1], "drho_k", 1e-4)
    _cmp(f[2], g[2], "Q", 1e-5)


@pytest.mark.parametrize("mech,nx,scheme", [
    ("h2_lidryer", 192, None), ("air5", 193, "weno7"), ("h2_lidryer", 512, None),
    ("air5", 513, None), ("h2_lidryer", 608, "weno7"), ("air5", 769, None)])
def test_x_lines_of_different_segments(mech, nx, scheme):
    """Lines that the convective sweep takes in other segments than the
    diffusive ones (more than 304 cells: at most 256 a segment against 304), and
    those whose cells end below the convective kernel's fixed 256 threads; the
    granular stage's bars of test_gpu_sweeps."""
    import flame3d_amd.abi as abi
    from test_gpu_sweeps import _cmp, _stage_pair
    sc = {"recon_kind": abi.RECON_WENO7} if scheme else None
    print(f"\n[x lines] {mech} nx={nx} {scheme}", flush=True)
    f, g = _stage_pair(mech, (nx, 4, 5), scheme=sc)
    _cmp(f[0], g[0], "dU", 1e-4)
    _cmp(f[1], g[1], "drho_k", 1e-4)
    _cmp(f[2], g[2], "Q", 1e-5)


@pytest.mark.parametrize("mech", ["air5", "h2_lidryer"])
def test_infinite_density(mech):
    """An infinite partial density leaves what does not depend on it as the
    oracle has it (its own D_k is a sum over the other species: 0), and an
    infinite density reads as an infinite pressure: a state that has run away
    does not turn into a small finite one."""
    import flame3d_amd.abi as abi
    import flame3d_amd.mech as mm
    from oracle import Oracle
    m = mm.load(mech)
    shape = (4, 4, 4)
    _, Q, rhoi = _state(shape, m)
    ctx, orc = abi.Context(*shape, m, "fp64"), Oracle(*shape, m)
    U = ctx.zeros(5)
    Qg, rg = Q.cuda(), rhoi.cuda()
    ctx.prim2c(U, Qg)
    rg[1, 7, 6, 5] = float("inf")
    out = [ctx.zeros(m.Ns), ctx.zeros(), ctx.zeros(), ctx.zeros(m.Ns)]
    ctx.mixture(Qg, rg, *out)
    torch.cuda.synchronize()
    ref = orc.mixture(to_np(Qg), to_np(rg))
    for got, want in zip(out, ref):
        assert np.allclose(to_np(got)[5, 6, 7], want[5, 6, 7], rtol=1e-12, atol=0, equal_nan=True)
    assert float(out[3][1, 7, 6, 5]) == 0.0
    rg = rhoi.cuda()
    U[0, 7, 6, 5] = float("inf")
    ctx.c2prim(U, Qg, rg)
    torch.cuda.synchronize()
    assert float(Qg[4, 7, 6, 5]) == float("inf")
    ctx.close()


@pytest.mark.parametrize("d", [0, 1, 2])
def test_single_species_has_no_diffusion_flux(d):
    """FP32 species faces: V_k - Y_k sum V is formed before it is multiplied by
    the enthalpy, so one species whose mass fraction at the face is one (0.75 and
    1.25 in turn along the sweep: a gradient, but a mean of 1) has no flux and
    carries no enthalpy: zero, not the rounding of two sums."""
    import flame3d_amd.abi as abi
    import flame3d_amd.cases as cases
    m = cases.tgv_gas()
    shape = (9, 8, 7)
    grid, Q, rhoi = _state(shape, m)
    ctx = abi.Context(*shape, m, "fp32")
    Q = Q.cuda()
    n = torch.arange(Q.shape[3 - d], device="cuda") % 2
    Y = (0.75 + 0.5 * n).float().reshape([-1 if 2 - d == k else 1 for k in range(3)])
    Y = Y.expand(Q.shape[1:]).contiguous()[None]
    D = ctx.rzeros(1) + 1e-4 * (1 + torch.rand(Q.shape[1:], device="cuda"))
    Fd, Fh = ctx.face_zeros(d, 1) + 1, ctx.face_zeros(d, 3) + 1
    ctx.spec_viscous_flux(d, Fd, Q, Y.contiguous(), [x.cuda() for x in grid.metrics],
                          grid.J.cuda(), D, Fh)
    torch.cuda.synchronize()
    assert int((Fd != 0).sum()) == 0 and int((Fh != 0).sum()) == 0
    ctx.close()


@pytest.mark.parametrize("shape,stretch,maxiter,slow_over", [
    ((48, 40, 36), 5.0, 3, 4096),        # all of a solve's iterations, more cells than may go
    ((112, 104, 96), 1.0, 50, None),     # a list of which one cell in 128 may go, and fewer do
    ((112, 104, 96), 5.0, 50, 8192),     # ... and more than that are slow
    ((144, 136, 136), 1.0, 50, None)])   # a list so long that no cell goes
def test_slow_cells_of_long_lists(shape, stretch, maxiter, slow_over):
    """Every rejected cell equals the Newton mode's bit for bit, whether the
    half-wave solve takes it, takes it on from a full list (from its beginning,
    or with two substeps at once where the first step failed) or takes none."""
    import flame3d_amd.abi as abi
    import flame3d_amd.cases as cases
    import flame3d_amd.mech as mm
    import flame3d_amd.surrogate as sur
    m = mm.load("h2_lidryer")
    print(f"\n[long list] {shape} dt x {stretch} maxiter {maxiter}", flush=True)
    Q, r = cases.chem_cells(shape, m, seed=7, dev="cuda")
    dt = stretch * sur.DT
    U = torch.zeros((5,) + tuple(Q.shape[1:]), dtype=torch.float64, device="cuda")
    ctx = abi.Context(*shape, m, "fp64")
    sur.attach(ctx, chain_max=1e-30, dt=dt)
    Un, Qn, rn = U.clone(), Q.clone(), r.clone()
    it = torch.zeros(shape[::-1], dtype=torch.int32, device="cuda")
    ctx.chem_newton(Un, Qn, rn, dt, maxiter, iters=it)
    st = torch.zeros(shape[::-1], dtype=torch.int8, device="cuda")
    n = int(ctx.nn_chem(U, Q, r, dt, maxiter, status=st))
    torch.cuda.synchronize()
    back = st >= 2
    slow = int((back & ((it > min(5, maxiter)) | (it < 0))).sum())
    print(f"[long list] {n} rejected, {slow} of them slow", flush=True)
    assert n == int(back.sum()) and n > st.numel() // 2
    if slow_over:
        assert slow > slow_over
    for got, ref in ((U, Un), (Q, Qn), (r, rn)):
        assert torch.equal(sur.interior(got)[back.flatten()], sur.interior(ref)[back.flatten()])
    ctx.close()


@pytest.mark.parametrize("a", [0, 1, 2, 3])
@pytest.mark.parametrize("b", [0, 1, 2, 3])
def test_fill_all_pairs(a, b):
    """All 16 ordered pairs of fill kinds of a direction's two faces, in each
    direction, on the smallest extents (4): with both faces in one launch, in
    turn, or one of them kept; equal bit for bit."""
    import flame3d_amd.abi as abi
    import flame3d_amd.mech as mm
    from oracle import Oracle
    m = mm.load("air5")
    shape = (4, 4, 4)
    _, Q, rhoi = _state(shape, m)
    orc, ctx = Oracle(*shape, m), abi.Context(*shape, m, "fp64")
    inQ = [1.2, 300.0, 1.0, -2.0, 1.0e5, 310.0, 2.0e5]
    inr = list(np.linspace(0.1, 0.2, m.Ns))
    for d in range(3):
        kinds = [2, 1, 1, 2, 3, 0]
        kinds[2 * d:2 * d + 2] = [a, b]
        Qo, ro = to_np(Q), to_np(rhoi)
        Uo = orc.prim2c(Qo)
        Qg, rg, Ug = Q.cuda(), rhoi.cuda(), to_torch(Uo)
        orc.fill(kinds, Qo, Uo, ro, inQ, inr)
        ctx.set_boundary(kinds, inQ, inr)
        ctx.fill(Qg, Ug, rg)
        torch.cuda.synchronize()
        for got, ref in ((Qg, Qo), (Ug, Uo), (rg, ro)):
            assert np.array_equal(to_np(got), ref), kinds
    ctx.close()


@pytest.mark.parametrize("shape", [(248, 248, 4), (249, 248, 5)])
def test_viscous_faces_at_the_plane_limit(shape):
    """FP64 viscous faces on the largest x-y plane that the y direction takes y
    by y (65536 points) and on one that it takes in slabs: 1e-12 normwise."""
    import flame3d_amd.abi as abi
    import flame3d_amd.mech as mm
    from oracle import Oracle
    m = mm.load("air5")
    grid, Q, rhoi = _state(shape, m)
    M, J = [to_np(x) for x in grid.metrics], to_np(grid.J)
    ctx, orc = abi.Context(*shape, m, "fp64"), Oracle(*shape, m)
    Qg, Mg, Jg = Q.cuda(), [x.cuda() for x in grid.metrics], grid.J.cuda()
    lam, mu = ctx.zeros() + 0.05, ctx.zeros() + 2e-5
    for d in range(3):
        Fv, Fh = ctx.face_zeros(d, 4), ctx.face_zeros(d, 3)
        ctx.viscous_flux(d, Fv, Qg, Mg, Jg, lam, mu, Fh)
        torch.cuda.synchronize()
        ref = orc.viscous_flux(d, to_np(Q), M, J, to_np(lam), to_np(mu), to_np(Fh))
        assert rel_err(to_np(Fv), ref) < 1e-12, d
    ctx.close()
