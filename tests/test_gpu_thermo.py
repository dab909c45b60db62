"""GPU subcycled cooling step against the reference fixtures and the oracle.

The GPU's rates use table-driven exp, log and pow (thermo_math.hpp), within an
ulp, and the reference glibc's; agreement is therefore to a tolerance, stated
per test."""
import os

import numpy as np
import pytest

from torch_amd import cooling_inputs

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _cooling(gpu, pfloor=None, **kw):
    p = gpu.thermo_params(**kw)
    if pfloor is not None:
        p.pfloor = pfloor
    return gpu.Cooling(p)


def test_thermo_params_match_oracle(gpu, orc):
    c = orc.converter(1e-20, 1e-28, 1e11)
    t = orc.thermo_params(c)
    p = gpu.thermo_params()
    for k in ("hydrogen_mass", "spec_gas_const", "dust_xsec", "imlc", "nmlc", "ciec", "n0", "nmc", "fuvh_a",
              "fuvh_b", "fuvh_c", "irh_a", "irh_b", "crh", "spl_min_slope", "spl_max_slope"):
        assert getattr(p, k) == getattr(t, k), k
    assert list(p.spl_y2) == list(t.spl_y2)


def test_thermo_cells_vs_reference_fixture(gpu):
    import torch

    f = np.load(os.path.join(GOLD, "thermo.npz"))
    inp = torch.from_numpy(np.ascontiguousarray(f["inputs"].T)).cuda()
    cool = _cooling(gpu, pfloor=float(f["pfloor"]))
    out, tot = cool.thermo_cells(inp)
    out = out.cpu().numpy()
    # heating and pre-step rate: one evaluation -> a few ulp of libm
    np.testing.assert_allclose(out[1], f["rate_pre"], rtol=1e-12, atol=0)
    ok = f["inputs"][:, 3] >= 1e-2
    np.testing.assert_allclose(out[0][ok], f["heat"][ok], rtol=1e-12, atol=0)
    # post-subcycle rate: after up to 2e5 explicit substeps, relative 1e-9
    rel = np.abs(out[2] - f["rate"]) / np.maximum(np.abs(f["rate"]), 1e-300)
    assert np.median(rel) < 1e-13
    assert np.quantile(rel, 0.999) < 1e-8, np.quantile(rel, [0.5, 0.99, 0.999, 1.0])


def test_thermo_cells_vs_oracle_workload_sample(gpu, orc):
    """Cells of the cooling workload (log-uniform rho, T, F, dt; uniform x,
    tau), including long subcycles; the subcycled pressure and the number of
    subcycles match the oracle."""
    import torch

    c = orc.converter(1e-20, 1e-28, 1e11)
    tc = lambda v, m, l, t: orc.to_code(c, v, m, l, t)  # noqa: E731
    s = cooling_inputs.sample_cgs(4096, seed=99)
    inp = cooling_inputs.to_code_inputs(s, tc)
    pfloor = 0.1 * tc(8.314462e7, 0, 2, -2) * tc(1e-30, 1, -3, 0) * 0.1
    t = orc.thermo_params(c, pfloor=pfloor)
    ref = orc.thermo_batch(t, inp, nthreads=8)
    cool = _cooling(gpu)
    assert cool.params.pfloor == pfloor
    out, tot = cool.thermo_cells(torch.from_numpy(np.ascontiguousarray(inp.T)).cuda())
    out = out.cpu().numpy()
    np.testing.assert_array_equal(out[3], ref[:, 3])          # subcycle counts
    assert tot == int(ref[:, 3].sum())
    rel = np.abs(out[4] - ref[:, 4]) / np.abs(ref[:, 4])      # subcycled pressure
    assert np.median(rel) < 1e-14 and rel.max() < 1e-6, np.quantile(rel, [0.5, 0.99, 1.0])


@pytest.mark.parametrize("knots", ["own", "lower", "between", "narrow", "wide", "uneven"])
def test_cooling_spline_takes_its_own_abscissae(gpu, orc, knots):
    """Spline tables whose abscissae are not the operator's own 3.5 .. 6.0:
    moved, of another spacing near 0.1, or uneven.  Pre-step rates of cells
    between 300 and 1e7 K against the oracle's bracketing search, both within
    a few ulp of log10 T on a spline of slope 60: 1e-12 of the terms."""
    import torch

    k = np.arange(26)
    x = {"own": None, "lower": 3.0 + 0.1 * k, "between": 3.55 + 0.1 * k, "narrow": 3.5 + 0.0985 * k,
         "wide": 3.4 + 0.1035 * k, "uneven": 3.5 + 0.1 * k + 0.04 * np.sin(2.1 * k)}[knots]
    c = orc.converter(1e-20, 1e-28, 1e11)
    tc = lambda v, m, l, t: orc.to_code(c, v, m, l, t)  # noqa: E731
    s = cooling_inputs.sample_cgs(4096, seed=21)
    inp = cooling_inputs.to_code_inputs(s, tc)
    T = 10.0 ** np.linspace(2.5, 7.0, 4096)
    inp[:, 1] = inp[:, 0] * tc(8.314462e7, 0, 2, -2) * (inp[:, 2] + 1.0) * T
    inp[:, 4] = inp[:, 1] / (1.67 - 1.0)
    t = orc.thermo_params(c, subcycling=False)
    p = gpu.thermo_params(subcycling=False)
    if x is not None:
        for i in range(26):
            t.spl_x[i] = p.spl_x[i] = x[i]
    p.pfloor = t.pfloor
    ref = orc.thermo_batch(t, inp, nthreads=8)
    out, _ = gpu.Cooling(p).thermo_cells(torch.from_numpy(np.ascontiguousarray(inp.T)).cuda())
    out = out.cpu().numpy()
    scale = np.abs(ref[:, 0]) + np.abs(ref[:, 1])
    err = np.abs(out[1] - ref[:, 1]) / scale
    assert err.max() < 1e-12, (err.max(), T[err.argmax()])


def test_uneven_spline_in_every_kernel(gpu, orc):
    """The kernels' instances for an uneven spline table: the integrator and the
    subcycle counts on cells that subcycle, against the oracle; the grid's time
    step and FP64 sub-step (inputs formed in the kernel) against the same on
    gathered inputs (heating record on)."""
    import torch

    from torch_amd import cloud
    from torch_amd import surrogate as sg

    k = np.arange(26)
    x = 3.5 + 0.1 * k + 0.04 * np.sin(2.1 * k)
    c = orc.converter(1e-20, 1e-28, 1e11)
    tc = lambda v, m, l, t: orc.to_code(c, v, m, l, t)  # noqa: E731
    p = gpu.thermo_params()
    t = orc.thermo_params(c, pfloor=p.pfloor)
    for i in range(26):
        t.spl_x[i] = p.spl_x[i] = x[i]
    inp = cooling_inputs.to_code_inputs(cooling_inputs.sample_cgs(2048, seed=5), tc)
    cool = gpu.Cooling(p)
    cnt = sg.subcycles(cool, torch.from_numpy(np.ascontiguousarray(inp.T)).cuda()).cpu().numpy()
    inp = np.ascontiguousarray(inp[(cnt >= 0) & (cnt <= 20000)])
    ref = orc.thermo_batch(t, inp, nthreads=8)
    dev = torch.from_numpy(np.ascontiguousarray(inp.T)).cuda()
    np.testing.assert_array_equal(sg.subcycles(cool, dev).cpu().numpy(), ref[:, 3])
    assert (ref[:, 3] > 8).sum() > 100
    out, _ = cool.thermo_cells(dev)
    rel = np.abs(out[4].cpu().numpy() - ref[:, 4]) / np.abs(ref[:, 4])
    assert np.median(rel) < 1e-14 and rel.max() < 1e-6, np.quantile(rel, [0.5, 0.99, 1.0])
    got = []
    for track in (False, True):
        gp, g, own, thermo = cloud.build(24, "fp64")
        Q = cloud.setup(24, tc)[0].copy()
        Q[1] *= 40.0    # 300 K to some 1e4 K, half ionised: the spline's term is the largest
        Q[2] = 0.5
        g.set_primitive(np.ascontiguousarray(Q))
        if track:
            g.heating_track(True)
        grid_p = gpu.thermo_params()
        grid_p.pfloor = gp.pfloor
        for i in range(26):
            grid_p.spl_x[i] = x[i]
        gc = gpu.Cooling(grid_p)
        dt = gc.grid_timestep(g, gp.dt_max, **thermo)
        assert dt != own.grid_timestep(g, gp.dt_max, **thermo)   # the table matters on this state
        gc.grid_substep(g, 100.0 * dt, **thermo)
        g.synchronize()
        got.append((dt, g.get_conserved()))
        g.close()
    assert got[0][0] == got[1][0]
    np.testing.assert_array_equal(got[0][1], got[1][1])


def test_cooling_rate_of_extreme_temperatures(gpu, orc):
    """Pre-step rates of neutral, half and fully ionised cells from 1e-300 to
    1e290 K (and some at the operator's own temperatures) against the
    oracle: ln T up to 690 times half an ulp in an exponent is 1e-13."""
    import torch

    c = orc.converter(1e-20, 1e-28, 1e11)
    t = orc.thermo_params(c, subcycling=False)
    p = gpu.thermo_params(subcycling=False)
    p.pfloor = t.pfloor
    T = np.concatenate([10.0 ** np.linspace(-300, 290, 1181), 10.0 ** np.linspace(1, 9, 161)])
    T, x = (a.ravel() for a in np.meshgrid(T, [0.0, 0.5, 1.0]))
    inp = np.zeros((T.size, 9))
    inp[:, 0] = 1e-10
    inp[:, 1] = inp[:, 0] * t.spec_gas_const * (x + 1.0) * T
    inp[:, 2], inp[:, 3], inp[:, 5] = x, 1.0, 100.0
    inp[:, 4] = inp[:, 1] / (1.67 - 1.0)
    inp[:, 8] = 1e-3
    ref = orc.thermo_batch(t, inp, nthreads=8)
    assert np.isfinite(ref[:, 1]).all()
    out, _ = gpu.Cooling(p).thermo_cells(torch.from_numpy(np.ascontiguousarray(inp.T)).cuda())
    out = out.cpu().numpy()
    err = np.abs(out[1] - ref[:, 1]) / (np.abs(ref[:, 0]) + np.abs(ref[:, 1]))
    assert err.max() < 1e-12, (err.max(), T[np.nanargmax(err)])


def test_infinite_rate_lands_softly(gpu, orc):
    """A cooling rate that overflows stays -inf within 200 K of the floor (as a
    division by 200 leaves it), and its subcycle count is refused."""
    import torch

    c = orc.converter(1e-20, 1e-28, 1e11)
    t = orc.thermo_params(c, subcycling=False)
    inp = np.zeros((64, 9))
    T = np.linspace(110.0, 500.0, 64)
    inp[:, 0], inp[:, 2], inp[:, 3], inp[:, 5], inp[:, 8] = 1e147, 0.5, 1.0, 100.0, 1e-3
    inp[:, 1] = inp[:, 0] * t.spec_gas_const * 1.5 * T
    inp[:, 4] = inp[:, 1] / (1.67 - 1.0)
    ref = orc.thermo_batch(t, inp, nthreads=1)
    assert (ref[:, 1] == -np.inf).all()
    dev = torch.from_numpy(np.ascontiguousarray(inp.T)).cuda()
    out, _ = _cooling(gpu, pfloor=t.pfloor, subcycling=False).thermo_cells(dev)
    np.testing.assert_array_equal(out[1].cpu().numpy(), ref[:, 1])
    with pytest.raises(gpu.TorchGpuError):
        _cooling(gpu, pfloor=t.pfloor).thermo_cells(dev)


def test_thermo_gate_and_no_subcycling(gpu, orc):
    import torch

    c = orc.converter(1e-20, 1e-28, 1e11)
    tc = lambda v, m, l, t: orc.to_code(c, v, m, l, t)  # noqa: E731
    inp = cooling_inputs.to_code_inputs(cooling_inputs.sample_cgs(512, seed=3), tc)
    inp[:256, 3] = 0.0  # ADV below thermo_hii_switch: exact no-op
    cool = _cooling(gpu, subcycling=False)
    out, _ = cool.thermo_cells(torch.from_numpy(np.ascontiguousarray(inp.T)).cuda())
    out = out.cpu().numpy()
    assert (out[2][:256] == 0).all() and (out[3] == 0).all()
    np.testing.assert_array_equal(out[2][256:], out[1][256:])  # RATE unchanged by integrate


def test_subcycle_counts_match_oracle(gpu, orc):
    """torchgpu_thermo_subcycles gives, without integrating, the number of
    subcycles Thermodynamics::integrate takes (Thermodynamics.cpp:303-312):
    equal to the oracle's count on cooling-workload cells and on cells of the
    cloud's conditions (dense, unlit, dt to 1e13 s), -1 where dt / dti is
    past the int range, and no error is left on the handle."""
    import torch

    from torch_amd import surrogate as sg

    c = orc.converter(1e-20, 1e-28, 1e11)
    tc = lambda v, m, l, t: orc.to_code(c, v, m, l, t)  # noqa: E731
    pfloor = 0.1 * tc(8.314462e7, 0, 2, -2) * tc(1e-30, 1, -3, 0) * 0.1
    t = orc.thermo_params(c, pfloor=pfloor)
    cool = _cooling(gpu)
    inp = cooling_inputs.to_code_inputs(cooling_inputs.sample_cgs(4096, seed=99), tc)
    cnt = sg.subcycles(cool, torch.from_numpy(np.ascontiguousarray(inp.T)).cuda()).cpu().numpy()
    ref = orc.thermo_batch(t, inp, nthreads=8)
    np.testing.assert_array_equal(cnt, ref[:, 3])
    # the cloud's conditions; one cell with dt / dti past the int range
    cl = cooling_inputs.to_code_inputs(cooling_inputs.sample_cgs_cloud(4096, seed=7), tc)
    cl[0, 8] = 1e300
    cnt = sg.subcycles(cool, torch.from_numpy(np.ascontiguousarray(cl.T)).cuda()).cpu().numpy()
    assert cnt[0] == -1 and (cnt >= -1).all()
    keep = (cnt >= 0) & (cnt <= 100000)
    assert keep.sum() > 2500 and (cnt[keep] > 4).sum() > 100, (keep.sum(), (cnt[keep] > 4).sum())
    ref = orc.thermo_batch(t, np.ascontiguousarray(cl[keep]), nthreads=8)
    np.testing.assert_array_equal(cnt[keep], ref[:, 3])
    # the counting call raised nothing: the integrator runs on the kept cells
    out, tot = cool.thermo_cells(torch.from_numpy(np.ascontiguousarray(cl[keep].T)).cuda())
    np.testing.assert_array_equal(out[3].cpu().numpy(), ref[:, 3])
