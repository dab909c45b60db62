"""GPU parity of the hydro step against the FP64 oracle (bitwise for FP64).

The oracle (oracle/torch_oracle.c) is itself pinned bitwise to the
reference's own translation units by tests/test_oracle_golden.py.
"""
import numpy as np
import pytest

from torch_amd import setups

pytestmark = pytest.mark.gpu


def _grid(gpu, shape, **kw):
    return gpu.Grid(gpu.make_params(shape, side_length=kw.pop("side_length", 1.0), **kw))


def _oparams(orc, shape, **kw):
    return orc.make_params(shape, kw.pop("dx"), nthreads=8, **kw)


def _u0(orc, p, Q):
    return orc.UfromQ_grid(orc.fix_primitives(p, Q, np.zeros_like(Q)), p.gamma)


def _run_both(gpu, orc, Q, nsteps, gkw=None, okw=None):
    gkw = gkw or {}
    okw = okw or {}
    shape = Q.shape[1:]
    g = _grid(gpu, shape, **gkw)
    g.set_primitive(np.ascontiguousarray(Q))
    p = _oparams(orc, shape, dx=gkw.get("side_length", 1.0) / shape[2], **okw)
    U0 = _u0(orc, p, Q)
    np.testing.assert_array_equal(g.get_conserved(), U0)
    g.run(nsteps)
    try:
        Uo, dts, t = orc.run_hydro(p, U0, nsteps)
    except RuntimeError as e:
        # the reference throws here; the GPU path must report the same error
        code = {"1": 3, "2": 4, "3": 5}[str(e).split("code ")[1].rstrip(")")]
        with pytest.raises(gpu.TorchGpuError) as ge:
            g.synchronize()
        assert ge.value.code == code, (ge.value, e)
        return None, None, None, None
    g.synchronize()
    Ug = g.get_conserved()
    tg, dtg, n = g.clock()
    return Ug, Uo, (tg, dtg, n), (t, dts[-1], nsteps)


@pytest.mark.parametrize("n,steps", [(16, 12), (32, 5)])
def test_sod_bitwise(gpu, orc, n, steps):
    Q = setups.sod(n)
    Ug, Uo, cg, co = _run_both(gpu, orc, Q, steps)
    np.testing.assert_array_equal(Ug, Uo)
    assert cg == co


@pytest.mark.parametrize("n,sigma,mach,steps", [(16, 1.0, 2.0, 20), (24, 1.5, 4.0, 10)])
def test_turbulent_bitwise(gpu, orc, n, sigma, mach, steps):
    Q = setups.turbulent(n, sigma, mach)
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12)
    Ug, Uo, cg, co = _run_both(gpu, orc, Q, steps, gkw=dict(kw), okw=dict(kw))
    np.testing.assert_array_equal(Ug, Uo)
    assert cg == co


@pytest.mark.parametrize("solver,limiter,order", [
    ("HLL", "minmod", 1), ("HLLC", "superbee", 1), ("RotatedHLLC", "monotonised_central", 1),
    ("RotatedHLLC", "leer", 1), ("HLLC", "ospre", 1), ("RotatedHLLC", "maxmod", 1), ("RotatedHLLC", "albada", 0)])
def test_solver_limiter_variants_ragged_grid(gpu, orc, solver, limiter, order):
    Q = setups.turbulent(16, 1.0, 1.5)[:, :9, :10, :12].copy()  # ragged 12 x 10 x 9
    bcs = ["outflow", "inflow", "periodic", "periodic", "reflecting", "free"]
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12, solver=solver, limiter=limiter,
              spatial_order=order, bc=bcs)
    Ug, Uo, cg, co = _run_both(gpu, orc, Q, 6, gkw=dict(kw), okw=dict(kw))
    np.testing.assert_array_equal(Ug, Uo)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("solver", ["HLL", "HLLC", "RotatedHLLC"])
def test_negative_face_pressure_raises(gpu, orc, solver, precision, axis):
    """maxmod takes the larger of two one-sided slopes, which a pressure jump of
    1 to 1,000 carries below zero at the face before it: the square of the sound
    speed there is negative and the flux is NaN, which the reference throws on
    and every solver of either precision reports."""
    Q = np.zeros((7, 12, 12, 12))
    Q[0], Q[1] = 1.0, 1.0
    Q[2], Q[3] = 0.5, 1.0
    P = np.moveaxis(Q[1], 2 - axis, 0)
    P[6], P[7:] = 1.1, 1000.0
    kw = dict(solver=solver, limiter="maxmod")
    p = _oparams(orc, (12, 12, 12), dx=1.0 / 12, **kw)
    with pytest.raises(RuntimeError) as e:
        orc.run_hydro(p, _u0(orc, p, Q), 1)
    assert "code 1" in str(e.value)
    g = _grid(gpu, (12, 12, 12), precision=gpu.MIXED if precision == "mixed" else gpu.FP64, **kw)
    g.set_primitive(Q)
    g.run(1)
    with pytest.raises(gpu.TorchGpuError) as ge:
        g.synchronize()
    assert ge.value.code == 3, ge.value


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_pure_hll_face_of_negative_pressure(gpu, orc, precision, axis):
    """As above, with two streams meeting along the axis at the jump: the
    rotated solver's normal is the axis, so its HLL solve, whose squared sound
    speed the velocity jump keeps positive, is all the face takes.  The mixed
    fluxes are sums of FP32 terms of the momentum flux's size (6^2 + 10 against
    a state of up to 34): 1e-4 of the largest value after two steps."""
    Q = np.zeros((7, 12, 12, 12))
    Q[0], Q[1] = 1.0, 1.0
    Q[2], Q[3] = 0.5, 1.0
    P, V = (np.moveaxis(Q[v], 2 - axis, 0) for v in (1, 4 + axis))
    P[6], P[7:] = 1.1, 10.0
    V[:6], V[6:] = 6.0, -6.0
    kw = dict(limiter="maxmod")
    p = _oparams(orc, (12, 12, 12), dx=1.0 / 12, **kw)
    ref, _, _ = orc.run_hydro(p, _u0(orc, p, Q), 2)
    g = _grid(gpu, (12, 12, 12), precision=gpu.MIXED if precision == "mixed" else gpu.FP64, **kw)
    g.set_primitive(Q)
    g.run(2)
    g.synchronize()
    U = g.get_conserved()
    if precision == "fp64":
        np.testing.assert_array_equal(U, ref)
    else:
        assert np.abs(U - ref).max() < 1e-4 * np.abs(ref).max()


# sizes on both sides of the two FP64 layouts' rule (8 x 4 x 4 tiles below about
# a quarter of a million cells, 16 x 16 columns marched along z above), none a
# multiple of a tile, a column or a column's planes
@pytest.mark.parametrize("nz,ny,nx", [(3, 5, 7), (21, 33, 18), (85, 91, 101), (4, 301, 323), (131, 70, 75)])
@pytest.mark.parametrize("solver,limiter,order,bcs", [
    ("RotatedHLLC", "albada", 1, ["periodic", "periodic", "reflecting", "outflow", "inflow", "reflecting"]),
    ("RotatedHLLC", "minmod", 1, ["reflecting", "inflow", "periodic", "periodic", "periodic", "periodic"]),
    ("HLLC", "albada", 0, ["free", "reflecting", "inflow", "free", "reflecting", "outflow"]),
    ("HLL", "leer", 1, ["outflow", "free", "outflow", "periodic", "free", "inflow"])])
def test_layouts_bitwise(gpu, orc, nz, ny, nx, solver, limiter, order, bcs):
    if min(nz, ny, nx) < 4 and "reflecting" in bcs:
        bcs = ["outflow" if b == "reflecting" else b for b in bcs]  # cells 1 and 2 of such an axis are read
    rng = np.random.Generator(np.random.PCG64(nx))
    z, y, x = np.meshgrid(*[np.arange(n) / n for n in (nz, ny, nx)], indexing="ij")
    Q = np.empty((7, nz, ny, nx))
    for v in range(7):
        k = rng.integers(1, 4, 3)
        Q[v] = np.sin(2 * np.pi * (k[0] * x + k[1] * y + k[2] * z) + v) + 0.1 * rng.standard_normal((nz, ny, nx))
    Q[:2] = np.exp(0.5 * Q[:2])
    Q[2:4] = 0.5 + 0.3 * Q[2:4]
    Q[4:, : nz // 2, : ny // 3] = 0.25  # a region of uniform flow: the solver's pure paths
    Q[5:, :, :, : nx // 4] = 0.0
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12, solver=solver, limiter=limiter,
              spatial_order=order, bc=bcs)
    Ug, Uo, cg, co = _run_both(gpu, orc, Q, 3, gkw=dict(kw), okw=dict(kw))
    assert Ug is not None
    np.testing.assert_array_equal(Ug, Uo)
    assert cg == co


# states partly outside the range of the quick divisions: velocities and
# fractions down to 1e-110 (below 2^-300, or with differences and products
# that are) from a middle plane on, in one corner, or everywhere in steps of
# 1e-12 (the march stops at them), thin gas, a cell wider than 2^64; a tile grid and two
# march grids with several pieces along z
@pytest.mark.parametrize("nz,ny,nx", [(9, 13, 18), (70, 85, 91), (131, 70, 75)])
@pytest.mark.parametrize("state", ["tails", "corner", "quiet", "thin", "wide"])
@pytest.mark.parametrize("solver", ["RotatedHLLC", "HLL"])
def test_quick_division_range_bitwise(gpu, orc, nz, ny, nx, state, solver):
    rng = np.random.Generator(np.random.PCG64(nz))
    Q = 0.5 + 0.3 * rng.random((7, nz, ny, nx))
    Q[4:] -= 0.65
    kw = dict(tfloor=1e-12, pfloor=1e-60, dfloor=1e-60, solver=solver, limiter="albada")
    gkw = dict(kw)
    if state == "tails":
        Q[2:, nz // 3 + 1:] *= 10.0 ** rng.uniform(-110.0, 0.0, Q[2:, nz // 3 + 1:].shape)
    elif state == "corner":
        Q[4:, -2:, -2:, -1:] = 1e-100
        Q[3, 0, 0, 0] = 1e-300
    elif state == "quiet":  # the solver's pure paths, and its choice between them
        Q[4:] *= 10.0 ** (-12.0 * rng.integers(0, 9, (1, nz, 1, 1)))
        Q[0], Q[1] = 1.0, 1.0
    elif state == "thin":
        Q[:2, nz // 2:, ny // 2:, :5] *= 1e-33
    else:
        gkw["side_length"] = 1e22
    Ug, Uo, cg, co = _run_both(gpu, orc, Q, 3, gkw=gkw, okw=dict(kw))
    assert Ug is not None
    np.testing.assert_array_equal(Ug, Uo)
    assert cg == co


def test_explicit_step_and_timestep(gpu, orc):
    Q = setups.turbulent(16, 1.0, 2.0)
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12)
    g = _grid(gpu, Q.shape[1:], **kw)
    g.set_primitive(Q)
    p = _oparams(orc, Q.shape[1:], dx=1.0 / 16, **kw)
    U = _u0(orc, p, Q)
    for _ in range(3):
        dt_o = orc.hydro_timestep(p, orc.fix_primitives(p, orc.q_from_u(p, U), U))
        dt_g = g.hydro_timestep()
        assert dt_g == dt_o
        g.hydro_step(dt_g)
        U = orc.hydro_step(p, U, dt_o)
        g.synchronize()
        np.testing.assert_array_equal(g.get_conserved(), U)
    Qg = g.get_primitive(fix=True)
    np.testing.assert_array_equal(Qg, orc.fix_primitives(p, orc.q_from_u(p, U), U))


def test_deterministic_rerun(gpu):
    Q = setups.turbulent(32, 1.0, 2.0)
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12)
    out = []
    for _ in range(2):
        g = _grid(gpu, Q.shape[1:], **kw)
        g.set_primitive(Q)
        g.run(8)
        g.synchronize()
        out.append(g.get_conserved())
        g.close()
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_nan_state_raises(gpu, precision):
    """A non-finite conserved value makes the reference's checkValues throw
    (Torch.cpp:420-443); the GPU path reports it at the next sync, and the
    run ends at the failing step as the reference's does."""
    Q = setups.sod(16)
    g = _grid(gpu, Q.shape[1:], precision=gpu.FP64 if precision == "fp64" else gpu.MIXED)
    g.set_primitive(Q)
    U = g.get_conserved()
    U[1, 3, 4, 5] = np.nan
    g.set_conserved(U)
    g.run(5)
    with pytest.raises(gpu.TorchGpuError) as e:
        g.synchronize()
    assert e.value.code in (4, 5)
    assert "(step 0)" in str(e.value)
    assert g.clock()[2] == 1


def test_invalid_order_rejected(gpu):
    with pytest.raises(gpu.TorchGpuError) as e:
        gpu.Grid(gpu.make_params((8, 8, 8), spatial_order=2))
    assert e.value.code == 6


def test_mixed_precision_close_to_fp64(gpu):
    Q = setups.turbulent(32, 1.0, 2.0)
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12)
    res = []
    for prec in (gpu.FP64, gpu.MIXED):
        g = _grid(gpu, Q.shape[1:], precision=prec, **kw)
        g.set_primitive(Q)
        g.run(20)
        g.synchronize()
        res.append(g.get_primitive(fix=False))
        g.close()
    d64, dmx = res[0][0], res[1][0]
    rel_l1 = np.abs(dmx - d64).sum() / np.abs(d64).sum()
    assert rel_l1 < 1e-5, rel_l1


@pytest.mark.parametrize("solver,limiter,order", [
    ("HLL", "minmod", 1), ("HLLC", "superbee", 1), ("RotatedHLLC", "albada", 1), ("RotatedHLLC", "leer", 1),
    ("RotatedHLLC", "albada", 0)])
def test_mixed_kernel_variants_ragged_grid(gpu, orc, solver, limiter, order):
    """The mixed-precision kernel (float reconstruction and flux, rotation-free
    hybrid solver, FP64 accumulation) on a ragged 12 x 10 x 9 grid with every
    boundary condition against the FP64 oracle: relative L1 of density and
    pressure below 1e-5 after 6 steps (FP32 rounding, ~1e-7 per step)."""
    Q = setups.turbulent(16, 1.0, 1.5)[:, :9, :10, :12].copy()
    bcs = ["outflow", "inflow", "periodic", "periodic", "reflecting", "free"]
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12, solver=solver, limiter=limiter,
              spatial_order=order, bc=bcs)
    g = _grid(gpu, Q.shape[1:], precision=gpu.MIXED, **kw)
    g.set_primitive(np.ascontiguousarray(Q))
    p = _oparams(orc, Q.shape[1:], dx=1.0 / Q.shape[3], **kw)
    Uo, dts, t = orc.run_hydro(p, _u0(orc, p, Q), 6)
    g.run(6)
    g.synchronize()
    Ug = g.get_conserved()
    for v in (0, 1):
        rel = np.abs(Ug[v] - Uo[v]).sum() / np.abs(Uo[v]).sum()
        assert rel < 1e-5, (v, rel)
    tg, dtg, n = g.clock()
    assert n == 6 and abs(tg - t) / t < 1e-5


# pieces of 2 and more planes with a shorter last one, a single plane, and a
# box whose pieces are longest; fields smooth along each axis, so no cell is
# left to chance
@pytest.mark.parametrize("nz,ny,nx", [(21, 20, 18), (1, 30, 17), (3, 5, 40), (67, 90, 150), (33, 129, 200)])
@pytest.mark.parametrize("solver", ["RotatedHLLC", "HLLC", "HLL"])
def test_mixed_pieces_along_z(gpu, orc, nz, ny, nx, solver):
    """Against the FP64 oracle after 4 steps: FP32 rounding of the fluxes (6
    faces, 2^-24 each) into 8 stages gives below 1e-5 in relative L1."""
    z, y, x = np.meshgrid(*[np.arange(n) / n for n in (nz, ny, nx)], indexing="ij")
    Q = np.empty((7, nz, ny, nx))
    for v in range(7):
        Q[v] = np.sin(2 * np.pi * (x + (v % 3) * y + (v % 2 + 1) * z) + v)
    Q[:2] = np.exp(0.5 * Q[:2])
    Q[2:4] = 0.5 + 0.3 * Q[2:4]
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12, solver=solver, bc=["periodic"] * 6)
    g = _grid(gpu, Q.shape[1:], precision=gpu.MIXED, **kw)
    g.set_primitive(Q)
    p = _oparams(orc, Q.shape[1:], dx=1.0 / nx, **kw)
    Uo, _, _ = orc.run_hydro(p, _u0(orc, p, Q), 4)
    g.run(4)
    g.synchronize()
    Ug = g.get_conserved()
    for v in (0, 1, 4, 5, 6):
        rel = np.abs(Ug[v] - Uo[v]).sum() / np.abs(Uo[v]).sum()
        assert rel < 1e-5, (v, rel)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_mixed_faces_of_equal_states_moving_apart(gpu, orc, axis):
    """A velocity jump along the face normal alone takes the hybrid solver's
    HLL path; with equal states and jump^2 = 8 c^2 the HLLC solve that has no
    weight there divides zero by zero, which must not reach the flux."""
    n = 20
    Q = np.empty((7, n, n, n))
    Q[0], Q[1], Q[2], Q[3] = 1.0, 1.0, 0.5, 0.25
    Q[4:] = 0.0
    c = np.sqrt(5.0 / 3.0)
    half = np.arange(n) >= n // 2
    shape = [1, 1, 1]
    shape[2 - axis] = n
    for k, scale in enumerate((1.0, 1.0 - 2.0 ** -22, 1.0 + 2.0 ** -22, 1.0 + 2.0 ** -23)):
        Q[4 + axis] = np.sqrt(2.0) * c * scale * np.where(half, 1.0, -1.0).reshape(shape)
        kw = dict(gamma=5.0 / 3.0, tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12)
        g = _grid(gpu, Q.shape[1:], precision=gpu.MIXED, **kw)
        g.set_primitive(Q)
        p = _oparams(orc, Q.shape[1:], dx=1.0 / n, **kw)
        Uo, _, _ = orc.run_hydro(p, _u0(orc, p, Q), 1)
        g.run(1)
        g.synchronize()
        np.testing.assert_allclose(g.get_conserved()[0], Uo[0], rtol=1e-5)
        g.close()


def test_mixed_kernel_interior_and_ring_columns(gpu, orc):
    """A 64 x 48 x 40 grid, large enough that the mixed kernel has columns
    whose x and y halos lie inside the grid (their loads skip the ghost
    mapping; 16 x 16 columns: 2 x 1 of them) beside boundary columns, with
    periodic, reflecting, outflow and inflow boundaries and 40 planes (three
    z blocks, the last one partial): relative L1 of density, energy and
    momenta against the FP64 oracle below 1e-5 after 4 steps."""
    from torch_amd import setups

    Q = setups.turbulent(64, 1.0, 1.5)[:, :40, :48, :64].copy()
    bcs = ["periodic", "periodic", "reflecting", "outflow", "inflow", "outflow"]
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12, bc=bcs)
    g = _grid(gpu, Q.shape[1:], precision=gpu.MIXED, **kw)
    g.set_primitive(np.ascontiguousarray(Q))
    p = _oparams(orc, Q.shape[1:], dx=1.0 / Q.shape[3], **kw)
    Uo, dts, t = orc.run_hydro(p, _u0(orc, p, Q), 4)
    g.run(4)
    g.synchronize()
    Ug = g.get_conserved()
    for v in (0, 1, 4, 6):
        rel = np.abs(Ug[v] - Uo[v]).sum() / np.abs(Uo[v]).sum()
        assert rel < 1e-5, (v, rel)


@pytest.mark.parametrize("solver,limiter", [("RotatedHLLC", "albada"), ("HLL", "ospre"), ("HLLC", "leer")])
def test_mixed_kernel_large_code_values(gpu, orc, solver, limiter):
    """Code units with pressures of 1e24 and velocities of 1e12 (the
    turbulent field with p x 1e24, v x 1e12, the gas constant x 1e24 so that
    temperatures are unchanged): the squares of the FP32 limiter and the HLL
    S_l S_r dU term would overflow FP32 there.  The mixed kernel must match
    the FP64 oracle on the scaled problem to the same 1e-5 relative L1 as on
    the unscaled one."""
    Q = setups.turbulent(16, 1.0, 1.5)[:, :9, :10, :12].copy()
    Q[1] *= 1e24
    Q[4:7] *= 1e12
    R = 8.314462e7 * 1e24
    kw = dict(tfloor=1e-12, pfloor=0.1 * R * 1e-30 * 1e-12, spec_gas_const=R, solver=solver, limiter=limiter,
              bc=["outflow", "inflow", "periodic", "periodic", "reflecting", "free"])
    g = _grid(gpu, Q.shape[1:], precision=gpu.MIXED, **kw)
    g.set_primitive(np.ascontiguousarray(Q))
    p = _oparams(orc, Q.shape[1:], dx=1.0 / Q.shape[3], **kw)
    Uo, dts, t = orc.run_hydro(p, _u0(orc, p, Q), 6)
    assert np.isfinite(Uo).all()
    g.run(6)
    g.synchronize()
    Ug = g.get_conserved()
    for v in (0, 1):
        rel = np.abs(Ug[v] - Uo[v]).sum() / np.abs(Uo[v]).sum()
        assert rel < 1e-5, (v, rel)


def test_sod64_200_steps_bitwise_vs_reference_fixture(gpu):
    """The 64^3 Sod configuration through 200 steps on the GPU FP64 path
    against tests/golden/sod64.npz, which the reference's own translation
    units wrote: one x-line at steps 1, 2, 10 and 200 (all lines of the
    planar problem must be identical) and every dt."""
    import os

    f = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "sod64.npz"))
    g = _grid(gpu, (64, 64, 64))
    g.set_primitive(np.ascontiguousarray(setups.sod(64)))
    dts = []
    for s in range(1, 201):
        g.run(1)
        _, dt, n = g.clock()
        assert n == s
        dts.append(dt)
        if s in (1, 2, 10, 200):
            U = g.get_conserved()
            np.testing.assert_array_equal(U[:, 0, 0, :], f[f"U_{s}"], err_msg=f"step {s}")
            assert (U == U[:, :1, :1, :]).all(), s
    np.testing.assert_array_equal(np.array(dts), f["dts"])


def test_mixed_kernel_64bit_addressing_path(gpu):
    """The mixed kernel addresses each state variable by a 32-bit byte offset
    below 2^29 cells and with 64-bit addresses above; TORCHGPU_ADDR64=1 (read
    when a grid is created) takes the 64-bit path on a small grid.  Only the
    addressing differs, so both give the same state bit for bit (ragged grid
    with every boundary condition, 6 steps)."""
    import os

    Q = np.ascontiguousarray(setups.turbulent(32, 1.0, 2.0)[:, :20, :27, :31])
    bcs = ["outflow", "inflow", "periodic", "periodic", "reflecting", "free"]
    kw = dict(tfloor=1e-12, pfloor=0.1 * 8.314462e7 * 1e-30 * 1e-12, bc=bcs)
    out = []
    for a64 in ("0", "1"):
        os.environ["TORCHGPU_ADDR64"] = a64
        try:
            g = _grid(gpu, Q.shape[1:], precision=gpu.MIXED, **kw)
        finally:
            os.environ.pop("TORCHGPU_ADDR64", None)
        g.set_primitive(Q)
        g.run(6)
        g.synchronize()
        out.append((g.get_conserved(), g.clock()))
        g.close()
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
