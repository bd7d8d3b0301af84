"""The device headers' per-cell arithmetic, compiled for the host with the
hardware's estimates stood in for by float-accurate ones, against the same
formulas in IEEE or extended precision."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "tests", "host_cpu")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("devnum") / "devnum.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-ffp-contract=off", "-fno-builtin", "-fPIC", "-shared",
                    "-I", os.path.join(HOST, "stub"), "-I", os.path.join(ROOT, "method_amd", "csrc"),
                    os.path.join(HOST, "device_numerics.cc"), "-o", out], check=True)
    return ctypes.CDLL(out)


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def secant_ieee(Z, SbSq, D, tauBar, gam):
    """getPrimitiveVarsSingleCell's recovery (srrmhd.cc:512-581) for one cell."""
    f64 = np.float64

    def residual(z):
        vsq = SbSq / (z * z)
        if vsq >= 1 or z < 0:
            return f64(1e6)
        W = 1 / np.sqrt(1 - vsq)
        rho = D / W
        h = z / (rho * W * W)
        p = (gam - 1) * (h - rho) / gam
        if rho < 0 or p < 0 or W < 1 or h < 0:
            return f64(1e6)
        return (1 - (gam - 1) / (W * W * gam)) * z + ((gam - 1) / (W * gam) - 1) * D - tauBar

    x0, x1 = f64(Z), f64(Z) + 1e-4
    f0, f1 = residual(x0), residual(x1)
    best, bestf = x0, f0
    for it in range(50):
        if abs(f0) < 1e-12:
            return x0, it
        x0, x1, f1 = x1 - f1 * (x1 - x0) / (f1 - f0), x0, f0
        f0 = residual(x0)
        if abs(f0) < abs(bestf):
            best, bestf = x0, f0
    return best, -1


@pytest.mark.parametrize("guess,tauBar", [(1e30, 3.0), (1e12, 1e30), (0.0, 3.0), (-0.0, 3.0), (-1.0, 3.0), (2.5, 3.0),
                                          (3.5, 3.0), (1e-3, 0.5), (np.nan, 3.0), (np.inf, 3.0), (2.0, np.nan)])
def test_secant_keeps_the_best_iterate(lib, guess, tauBar):
    """A cell whose secant fails keeps its best iterate: an undefined residual
    (a NaN iterate) never takes its place, however large the best one's is. The
    same root, step count and failures as in IEEE arithmetic; a root found to
    |residual| < 1e-12 agrees to 1e-11 (the residual's slope in Z is above 0.1)."""
    rng = np.random.default_rng(3)
    n, gam = 50, 5.0 / 3.0
    SbSq, D = rng.uniform(0.1, 2.0, n), rng.uniform(0.2, 1.0, n)
    tb = np.full(n, tauBar)
    Z, its = np.full(n, guess), np.zeros(n, np.int32)
    lib.secant(n, ptr(SbSq), ptr(D), ptr(tb), ctypes.c_double(gam), ptr(Z), ptr(its))
    with np.errstate(all="ignore"):
        for k in range(n):
            z, it = secant_ieee(np.float64(guess), SbSq[k], D[k], tb[k], gam)
            assert (its[k] < 0) == (it < 0), (k, its[k], it)
            if np.isfinite(z):
                assert abs(Z[k] - z) <= 1e-11 * max(1.0, abs(z)), (k, Z[k], z)
            else:
                assert np.array_equal(Z[k], z, equal_nan=True), (k, Z[k], z)


EPS = 2.0 ** -53  # one rounding


def cold_states(n, ratio, W, seed):
    """rho, p, v, B of n states with p / rho about `ratio` and Lorentz factors up to W."""
    rng = np.random.default_rng(seed)
    rho = np.exp(rng.uniform(np.log(0.1), np.log(10.0), n))
    p = rho * ratio * rng.uniform(0.5, 1.5, n)
    v = rng.normal(size=(3, n))
    v *= np.sqrt(1 - 1 / (1 + (W - 1) * rng.uniform(0.01, 1.0, n)) ** 2) / np.sqrt((v * v).sum(0))
    return rho, p, v, rng.normal(size=(3, n)) * 0.3 * np.sqrt(rho)


@pytest.mark.parametrize("ratio", [1.0, 1e-3, 1e-4, 1e-6])
@pytest.mark.parametrize("W", [1.2, 5.0, 50.0])
def test_recovery_rounds_h_once(lib, ratio, W):
    """rho and h from a given root against extended precision, and p, which in a
    cold cell is what is left of h - 1. With s = 1 - v^2 a rounding of at most
    1/2 in sqrt(s), sqrt(s), its product and the quotient one each, h is within
    3.5 roundings (3 more of the rsqrt's would not be) and 1.5 on average (four
    uniform errors add to 0.5 on average), rho within 2.5; p = (h - 1) rho (gam -
    1) / gam adds four to h's, weighed by h / (h - 1), and e as many."""
    n, gam = 20000, 5.0 / 3.0
    rho, p, v, B = cold_states(n, ratio, W, 5)
    v2 = (v * v).sum(0)
    Z = (rho + p * gam / (gam - 1)) / (1 - v2)
    U = np.ascontiguousarray(np.concatenate([[rho / np.sqrt(1 - v2)], Z * v, [Z], B, 0 * rho[None]]).T)
    root = np.ascontiguousarray(np.stack([v2, Z], 1))
    P, A = np.zeros((n, 8)), np.zeros((n, 13))
    lib.recover(n, ptr(U), ptr(root), ctypes.c_double(gam), ptr(P), ptr(A))
    L = np.longdouble
    iW = np.sqrt(1 - L(v2))
    r, h = L(U[:, 0]) * iW, L(Z) * iW / L(U[:, 0])
    check_recovered(P[:, 0], P[:, 4], A[:, 0], r, (h - 1) * r * (L(gam) - 1) / L(gam), h)


def check_recovered(rho, p, h, r, q, H):
    def err(x, y):
        return np.abs((x - y) / y).astype(float) / EPS

    assert err(h, H).max() <= 3.6 and err(h, H).mean() <= 1.0
    assert err(rho, r).max() <= 2.6
    weight = (H / (H - 1)).astype(float)
    assert (err(p, q) / (4 + 3.6 * weight)).max() <= 1.0
    assert (err(p, q) / (4 + weight)).mean() <= 1.0


@pytest.mark.parametrize("ratio", [1.0, 1e-3, 1e-6])
@pytest.mark.parametrize("W", [1.2, 5.0])
def test_resistive_recovery_rounds_h_once(lib, ratio, W):
    """The same for the resistive model, whose root is Z alone: v^2 = Sbar^2 / Z^2
    takes two more roundings, which W^2 v^2 / 2 weighs in 1/W; the states here have
    Sbar along x alone (E = 0), so h is within 3.5 + W^2 roundings."""
    n, gam = 20000, 5.0 / 3.0
    rho, p, v, B = cold_states(n, ratio, W, 6)
    v2 = (v * v).sum(0)
    Z = (rho + p * gam / (gam - 1)) / (1 - v2)
    zero = 0 * rho
    U = np.ascontiguousarray(np.stack([rho / np.sqrt(1 - v2), Z * np.sqrt(v2), zero, zero, Z] + [zero] * 9, 1))
    P, A = np.zeros((n, 11)), np.zeros((n, 17))
    lib.recover_resistive(n, ptr(U), ptr(Z), ctypes.c_double(gam), ctypes.c_double(10.0), ptr(P), ptr(A))
    L = np.longdouble
    vsq = (L(U[:, 1]) / L(Z)) ** 2
    iW = np.sqrt(1 - vsq)
    h = L(Z) * iW / L(U[:, 0])

    def err(x, y):
        return np.abs((x - y) / y).astype(float) / EPS

    W2 = (1 / (1 - vsq)).astype(float)
    assert (err(A[:, 0], h) / (3.6 + W2)).max() <= 1.0
    e = (L(A[:, 0]) - 1) / L(gam)  # e and p from the h and rho that were returned: five roundings at most
    assert err(P[:, 4], L(P[:, 0]) * e * (L(gam) - 1)).max() <= 5.0
    assert err(A[:, 9], vsq).max() <= 3.1  # Sbar^2, Z^2 and the quotient


def test_refined_rsqrt_is_one_rounding(lib):
    """1 / sqrt(b) is rounded once (the refinement leaves e^3 = 2^-69 and products
    of roundings with the estimate's 2^-24). With the root, the root is rounded
    once and the other is its reciprocal, rounded once more."""
    rng = np.random.default_rng(1)
    b = np.concatenate([rng.uniform(0, 1, 200000), 2.0 ** rng.uniform(-60, 60, 200000), [1.0, 0.25, 2.0 ** -53]])
    alone, w, root = (np.zeros_like(b) for _ in range(3))
    lib.rsqrt_refined(b.size, ptr(b), ptr(alone), ptr(w), ptr(root))
    L = np.longdouble
    exact = np.sqrt(L(b))
    assert (np.abs(alone * exact - 1) / EPS).max() <= 1.01
    assert (np.abs(root / exact - 1) / EPS).max() <= 1.01
    assert (np.abs(w * L(root) - 1) / EPS).max() <= 1.01


@pytest.mark.parametrize("ratio", [1.0, 1e-3])
@pytest.mark.parametrize("W", [1.2, 5.0])
def test_flux_error_is_that_of_ieee_operations(lib, ratio, W):
    """The flux of S and tau with the refined 1/W and W against the same sums with
    an IEEE square root and division, both against extended precision: the mean
    error, in parts of the flux vector's length, is the same to the 3 % that
    20,000 states leave it uncertain."""
    n, gam = 20000, 5.0 / 3.0
    rho, p, v, B = cold_states(n, ratio, W, 7)
    v2 = (v * v).sum(0)
    e = (rho + p * gam / (gam - 1)) / (1 - v2)
    U = np.ascontiguousarray(np.concatenate([[rho / np.sqrt(1 - v2)], e * v, [e - p], B, 0 * rho[None]]).T)
    P = np.ascontiguousarray(np.concatenate([[rho], v, [p], B]).T)
    got, ieee = np.zeros((n, 4)), np.zeros((n, 4))
    lib.flux_x(n, ptr(U), ptr(P), ptr(got))
    lib.flux_x_ieee(n, ptr(U), ptr(P), ptr(ieee))
    L = np.longdouble
    u, w, b = L(U), L(P[:, 1:4]), L(U[:, 5:8])
    iW = np.sqrt(1 - (w * w).sum(1))
    b0 = (w * b).sum(1) / iW
    ptot = L(P[:, 4]) + ((b * b).sum(1) + b0 * b0) * iW * iW / 2
    exact = u[:, 1:5] * w[:, :1]
    exact[:, :3] -= (b * iW[:, None] + b0[:, None] * w) * (b[:, 0] * iW)[:, None]
    exact[:, 0] += ptot
    exact[:, 3] += ptot * w[:, 0] - b0 * b[:, 0] * iW
    size = np.sqrt((exact * exact).sum(1))[:, None]
    mean = [(np.abs(x - exact) / size).astype(float).mean(0) for x in (got, ieee)]
    assert (mean[0] <= 1.03 * mean[1]).all(), (mean[0] / EPS, mean[1] / EPS)


@pytest.mark.gpu
@pytest.mark.parametrize("resistive", [False, True])
def test_recovered_density_and_lorentz_factor_on_the_device(resistive):
    """With the hardware's own estimates: 1/W is D's factor in rho and W its
    reciprocal, rounded once each, so rho W gives D back to two roundings."""
    from method_amd import engine as eng
    from method_amd import initdata as idt

    n, ng = 96, 4
    g = idt.Grid(n, n, 0, -0.5, 0.5, -1.0, 1.0)
    p = idt.kh_prims(g, seed=2)
    p[4] *= 1e-3
    cfg = dict(model=eng.SRMHD, integrator=eng.RK2)
    if resistive:
        p = np.concatenate([p, -np.cross(p[1:4], p[5:8], axis=0)])
        cfg = dict(model=eng.SRRMHD, integrator=eng.SSP2, sigma=10.0)
    print(f"gpu: rho W = D, resistive={resistive}", flush=True)
    with eng.Engine(eng.Config(n, n, 0, -0.5, 0.5, -1.0, 1.0, **cfg)) as e:
        e.set_prims(p)
        for _ in range(3):
            e.update_time()
        c, q, a = (x[:, ng:-ng, ng:-ng] for x in e.download())
    assert np.isfinite(q).all()
    assert (np.abs(np.longdouble(q[0]) * a[1] / c[0] - 1) / EPS).max() <= 2.05
