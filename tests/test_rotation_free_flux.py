"""The mixed-precision kernel evaluates the rotated hybrid HLLC-HLL flux
without rotation matrices (hydro_math.hpp, riemann_f): solving along a unit
normal n in the original frame with u_n = v.n, and n2 = (d - n1_d n1) / s; and
it sums the two solvers' fluxes as scalars (NormalFlux: a mass flux per side, a
conserved jump, a pressure term along the normal and the energy flux) before it
forms the one flux vector.  This test restates that in float64 numpy, the
combination line for line, and checks it against the oracle's literal
rotate-solve-rotate-back solver (Riemann.cpp:154-244) on the
reference-derived KAT inputs of tests/golden/riemann.npz: the two must agree
to rounding (the identity is exact in real arithmetic), so a wrong sign of n2,
a dropped pressure term or jump, or a wrong star-state velocity fails it."""
import os

import numpy as np
import pytest

import oracle

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
DEN, PRE, HII, ADV, VEL = 0, 1, 2, 3, 4


def _side(q, g):
    rho, p, v = q[:, DEN], q[:, PRE], q[:, VEL:VEL + 3]
    ke = 0.5 * rho * (v * v).sum(1)
    return dict(rho=rho, p=p, x=q[:, HII], a=q[:, ADV], v=v, sr=np.sqrt(rho), a2=g * p / rho, ke=ke,
                E=p / (g - 1.0) + ke)


def _speeds(L, R, unl, unr):
    is_ = 1.0 / (L["sr"] + R["sr"])
    ut = (L["sr"] * unl + R["sr"] * unr) * is_
    d = np.sqrt((L["sr"] * L["a2"] + R["sr"] * R["a2"]) * is_ + 0.5 * L["sr"] * R["sr"] * is_ * is_ * (unr - unl) ** 2)
    return ut - d, ut + d


def _hll(L, R, unl, unr, g2):
    """(hl, hr, s, c, e) of the HLL flux along a normal."""
    Sl, Sr = _speeds(L, R, unl, unr)
    wr = np.clip(Sr / (Sr - Sl), 0.0, 1.0)
    wl = 1.0 - wr
    hl, hr, s = wr * unl, wl * unr, np.minimum(Sl, 0.0) * wr
    e = hl * (g2 * L["p"] + L["ke"]) + hr * (g2 * R["p"] + R["ke"]) + s * (R["E"] - L["E"])
    return hl, hr, s, wr * L["p"] + wl * R["p"], e


def _hllc(L, R, unl, unr, g2):
    Sl, Sr = _speeds(L, R, unl, unr)
    wl, wr = L["rho"] * (Sl - unl), R["rho"] * (Sr - unr)
    Sc = (R["p"] - L["p"] + wl * unl - wr * unr) / (wl - wr)
    sub = ~(Sl >= 0) & ~(Sr <= 0)
    left = (Sl >= 0) | (sub & (Sc >= 0))
    rho, p, E = (np.where(left, L[k], R[k]) for k in ("rho", "p", "E"))
    un, S = np.where(left, unl, unr), np.where(left, Sl, Sr)
    iss = np.where(sub, 1.0 / np.where(sub, S - Sc, 1.0), 0.0)
    wi = (S - un) * iss
    t = np.where(sub, wi * Sc, un)
    dsc = np.where(sub, Sc - un, 0.0)
    sd = S * dsc
    e = t * E + p * (un + sd * iss) + sd * (rho * t)
    return np.where(left, t, 0.0), np.where(left, 0.0, t), np.zeros_like(t), p + sd * (rho * wi), e


def normal_flux(solver, Ql, Qr, dims, g):
    """Flux along axis dims[i] of each face as riemann_f forms it."""
    L, R = _side(Ql, g), _side(Qr, g)
    g2 = g / (g - 1.0)
    i = np.arange(Ql.shape[0])
    D, A, B = dims, np.where(dims == 0, 1, 0), np.where(dims == 2, 1, 2)
    lv, rv = L["v"], R["v"]
    zero = np.zeros(i.size)
    nA = nB = ct = zero
    if solver != "RotatedHLLC":
        hl, hr, sj, cd, e = (_hll if solver == "HLL" else _hllc)(L, R, lv[i, D], rv[i, D], g2)
    else:
        nd, nA, nB = (rv[i, X] - lv[i, X] for X in (D, A, B))
        nn = nd * nd + nA * nA + nB * nB
        small = nn < 1.0e-12
        n = np.where(small, 0.0, np.copysign(1.0 / np.sqrt(np.where(small, 1.0, nn)), nd))
        nA, nB = nA * n, nB * n
        s2 = nA * nA + nB * nB
        axis = s2 == 0.0
        nd = np.where(axis, 1.0, nd * n)
        is_ = 1.0 / np.sqrt(np.where(axis, 1.0, s2))
        s = np.where(axis, np.where(small, 1.0, 0.0), s2 * is_)
        k = np.where(axis, 0.0, nd * is_)
        ql, qr = lv[i, A] * nA + lv[i, B] * nB, rv[i, A] * nA + rv[i, B] * nB
        f1 = _hll(L, R, nd * lv[i, D] + ql, nd * rv[i, D] + qr, g2)
        f2 = _hllc(L, R, s * lv[i, D] - k * ql, s * rv[i, D] - k * qr, g2)
        w1 = np.where(small, 0.0, nd)
        hl, hr, sj = w1 * f1[0] + s * f2[0], w1 * f1[1] + s * f2[1], w1 * f1[2]
        e = w1 * f1[4] + s * f2[4]
        c1, c2 = w1 * f1[3], s * f2[3]
        cd, ct = c1 * nd + c2 * s, c1 - c2 * k
    ml, mr = L["rho"] * hl, R["rho"] * hr

    def flux(l, r, c=zero):
        return ml * l + (mr * r + (sj * (R["rho"] * r - L["rho"] * l) + c))

    F = np.empty((i.size, 7))
    F[:, DEN] = ml + mr + sj * (R["rho"] - L["rho"])
    F[:, PRE] = e
    F[:, HII], F[:, ADV] = flux(L["x"], R["x"]), flux(L["a"], R["a"])
    for X, c in ((D, cd), (A, ct * nA), (B, ct * nB)):
        F[i, VEL + X] = flux(lv[i, X], rv[i, X], c)
    return F


@pytest.mark.parametrize("solver", ["RotatedHLLC", "HLL", "HLLC"])
def test_rotation_free_matches_rotated_solver(solver):
    f = np.load(os.path.join(GOLD, "riemann.npz"))
    Ql, Qr, dims, g = f["Ql"], f["Qr"], f["dims"].astype(int), float(f["gamma"])
    ref, st = oracle.riemann(solver, Ql, Qr, dims, g)
    ok = st == 0
    got = normal_flux(solver, Ql, Qr, dims, g)
    # relative to the face's flux scale (momentum flux ~ p + rho v^2)
    scale = np.abs(ref[ok]).max(1, keepdims=True) + 1e-300
    err = np.abs(got[ok] - ref[ok]) / scale
    assert np.isfinite(got[ok]).all()
    assert np.median(err) < 1e-14, np.median(err)
    assert err.max() < 1e-9, (err.max(), np.argmax(err.max(1)))
