"""The FP64 sweeps' common path (riemann_hlld_lean, riemann_hllx_lean) against the full solver
it replaces and against the oracle, interface by interface. rmhd_device.hpp is compiled for
the host with stand-ins for the hardware approximations (tests/host)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HLL, HLLC, HLLD = 0, 1, 2
DEFER = 100
DOUBLES, INTS = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)


class Solvers:
    def __init__(self, path):
        self.lib = ctypes.CDLL(path)

    def __call__(self, which, solver, PL, PR, gamma=4.0 / 3.0, pfloor=0.0):
        """Flux, return code, fastest speed and p* steps of n interfaces normal to x."""
        PL, PR = np.ascontiguousarray(PL, dtype=float), np.ascontiguousarray(PR, dtype=float)
        n = len(PL)
        F, lam, rc, steps = np.zeros((n, 8)), np.zeros(n), np.zeros(n, np.int32), np.zeros(n, np.int32)
        getattr(self.lib, which)(ctypes.c_int(solver), ctypes.c_long(n), PL.ctypes.data_as(DOUBLES),
                                 PR.ctypes.data_as(DOUBLES), ctypes.c_double(gamma), ctypes.c_double(pfloor),
                                 F.ctypes.data_as(DOUBLES), rc.ctypes.data_as(INTS), lam.ctypes.data_as(DOUBLES),
                                 steps.ctypes.data_as(INTS))
        return F, rc, lam, steps


    def side_flux(self, P, gamma=4.0 / 3.0):
        P = np.ascontiguousarray(P, dtype=float)
        F, G = np.zeros_like(P), np.zeros_like(P)
        self.lib.side_flux(ctypes.c_long(len(P)), P.ctypes.data_as(DOUBLES), ctypes.c_double(gamma),
                           F.ctypes.data_as(DOUBLES), G.ctypes.data_as(DOUBLES))
        return F, G

    def plm_ahead(self, V, theta):
        V = np.ascontiguousarray(V, dtype=float)
        out = [np.zeros(len(V), t) for t in (np.float64, np.float64, np.float32, np.float32)]
        self.lib.plm_ahead(ctypes.c_long(len(V)), V.ctypes.data_as(DOUBLES), ctypes.c_double(theta),
                           *(o.ctypes.data_as(ctypes.c_void_p) for o in out))
        return out

    def weno5(self, V):
        V = np.ascontiguousarray(V, dtype=float)
        F, G = np.zeros((len(V), 4)), np.zeros((len(V), 4))
        self.lib.weno5(ctypes.c_long(len(V)), *(a.ctypes.data_as(DOUBLES) for a in (V, F, G)))
        return F, G


@pytest.fixture(scope="module")
def solvers(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "solvers.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=fast", "-fopenmp", "-w", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "tests", "host"), "-I", os.path.join(ROOT, "ctf_amd", "csrc"),
                    "-o", out, os.path.join(ROOT, "tests", "host", "solvers.cpp")], check=True)
    return Solvers(out)


# interfaces whose right fast wave moves left while the right Alfven wave moves right
TRANS_FAST = [
    ([6.2163, 0.46995, -0.2378, -0.7187, -0.473, 2.0485, 0.7083, -1.1451],
     [8.0491, 0.24608, -0.55881, -0.41229, -0.21378, 2.0485, 1.3851, -0.22483]),
    ([1.0805, 0.28644, -0.54631, 0.59338, -0.31491, 1.6803, 0.13063, -1.4054],
     [1.1193, 0.1588, -0.65694, 0.10161, -0.53991, 1.6803, -0.89298, 0.2466]),
    ([0.88341, 0.044542, -0.44481, 0.66776, -0.22813, -0.82136, 0.11297, 0.32027],
     [0.34259, 0.023266, -0.66294, 0.21559, -0.52903, -0.82136, 0.48395, -0.17018]),
    ([1.8798, 0.37374, -0.50156, 0.52429, 0.048764, -0.84443, 0.44374, 0.26674],
     [1.0173, 0.17073, -0.40034, -0.11127, 0.5813, -0.84443, 0.080919, 0.052828]),
    ([0.60645, 0.058776, -0.74339, -0.34436, -0.26366, 1.0373, -0.44309, 0.87441],
     [0.3555, 0.030151, -0.75145, -0.36283, 0.20616, 1.0373, 0.18288, -0.027719]),
    ([1.0031, 0.33669, -0.53523, -0.57094, 0.30507, -1.9073, 0.75086, -0.075821],
     [0.8959, 0.1353, -0.79157, -0.26121, 0.22481, -1.9073, -0.10198, 0.063667]),
    ([0.37575, 0.053587, -0.55838, -0.35888, -0.63519, 1.291, -0.17125, -0.28025],
     [0.41098, 0.028817, -0.6138, -0.018785, -0.65501, 1.291, -0.21529, 0.046615]),
]


def test_trans_fast_fan(solvers, oracle_lib):
    """HLLD accepts fans whose right fast wave lies left of the right Alfven wave; the wave chain
    asks for the contact and the Alfven waves before the right fast wave
    (Mara/riemann_hlld-rmhd.cpp:518-524), so s = 0 between them takes the state there and not
    the right state. The flux of every interface that the common path keeps against the full
    solver and the oracle, 1e-10 of its largest component."""
    PL, PR = (np.array(side) for side in zip(*TRANS_FAST))
    F, rc, _, _ = solvers("lean", HLLD, PL, PR)
    G, full_rc, _, _ = solvers("full", HLLD, PL, PR)
    O = np.array([oracle_lib.riemann("hlld", l[None], r[None], 1, 4.0 / 3.0)[0][0] for l, r in zip(PL, PR)])
    assert (full_rc == 0).all() and np.isin(rc, (0, DEFER)).all()
    scale = np.abs(G).max(axis=1, keepdims=True)
    assert (np.abs(G - O) <= 1e-10 * scale).all()
    keep = rc == 0
    assert (np.abs(F - G)[keep] <= 1e-10 * scale[keep]).all()


def random_interfaces(rng, n, jump, W, beta):
    """Interfaces with jumps of the given size between states with Lorentz factors up to W and
    fields of the order of beta (log-normal), the normal field continuous."""
    P = np.empty((n, 8))
    P[:, 0] = np.exp(rng.normal(0.0, 1.0, n))
    P[:, 1] = P[:, 0] * np.exp(rng.normal(-0.5, 1.2, n))
    e = rng.normal(size=(n, 3))
    w = 1.0 + (W - 1.0) * rng.uniform(0, 1, n)
    P[:, 2:5] = e / np.linalg.norm(e, axis=1)[:, None] * np.sqrt(1.0 - w ** -2.0)[:, None]
    P[:, 5:8] = beta * rng.normal(size=(n, 3)) * np.exp(rng.normal(-0.5, 1.0, n))[:, None]
    Q = P.copy()
    Q[:, :2] *= np.exp(jump * rng.uniform(-1, 1, (n, 2)))
    u = P[:, 2:5] * w[:, None] + jump * rng.uniform(-1, 1, (n, 3))
    Q[:, 2:5] = u / np.sqrt(1.0 + (u * u).sum(axis=1))[:, None]
    Q[:, 5:8] += jump * np.abs(P[:, 5:8]).max(axis=1)[:, None] * rng.uniform(-1, 1, (n, 3))
    Q[:, 5] = P[:, 5]
    return P, Q


@pytest.mark.parametrize("solver", [HLLD, HLLC, HLL])
@pytest.mark.parametrize("beta", [0.1, 1.0, 3.0])
def test_kept_interfaces_have_the_full_solvers_flux(solvers, solver, beta):
    """What the common path keeps is what the full solver decides, also where the full p* solve
    is at the end of its reach (many steps, a residual whose round-off is near its tolerance)
    and falls to another attempt or to HLLC. 600 000 random interfaces: at most one kept
    interface in 100 000 off by more than 1e-9 of its flux (some are so ill-conditioned
    that round-off does it). Without a rule for such solves 1 in 600 of the HLLD ones are at
    beta = 3, and 1 in 7 000 at beta = 1."""
    rng = np.random.default_rng(12)
    kept = off = 0
    for jump in (1e-3, 0.02, 0.1, 0.3, 1.0):
        for W in (1.05, 1.5, 3.0):
            PL, PR = random_interfaces(rng, 40000, jump, W, beta)
            F, rc, _, _ = solvers("lean", solver, PL, PR)
            G, full_rc, _, _ = solvers("full", solver, PL, PR)
            assert np.isin(rc, (0, DEFER)).all()
            keep = rc == 0
            assert (full_rc[keep] == 0).all()
            d = np.abs(F - G).max(axis=1) / np.abs(G).max(axis=1)
            kept += keep.sum()
            off += (keep & ~(d <= 1e-9)).sum()
    assert kept > 400000
    assert off <= 1e-5 * kept


def cold_or_empty(rng, n, kind):
    """Interfaces at the edge of what prim_to_cons takes: an internal energy within round-off of
    the rest mass's, no density, or a pressure below zero."""
    P = np.zeros((n, 8))
    P[:, 0] = 0.0 if kind == "empty" else np.exp(rng.normal(0, 2, n))
    if kind == "cold":
        P[:, 1] = P[:, 0] * 10 ** rng.uniform(-19, -13, n)
        P[:, 2:5] = rng.normal(size=(n, 3)) * 10 ** rng.uniform(-10, -6, (n, 1))
        P[:, 5:8] = rng.normal(size=(n, 3)) * 10 ** rng.uniform(-10, -7, (n, 1))
    else:
        P[:, 1] = 10 ** rng.uniform(-3, 0, n) * (1.0 if kind == "empty" else -P[:, 0])
        P[:, 2:5] = 0.5 * rng.uniform(-1, 1, (n, 3))
        P[:, 5:8] = rng.normal(size=(n, 3))
    Q = P * (1 + 1e-3 * rng.uniform(-1, 1, P.shape))
    Q[:, 5] = P[:, 5]
    return P, Q


@pytest.mark.parametrize("solver", [HLLD, HLLC, HLL])
@pytest.mark.parametrize("kind", ["cold", "empty", "negative pressure"])
def test_what_the_full_solver_refuses_is_not_kept(solvers, solver, kind):
    PL, PR = cold_or_empty(np.random.default_rng(2), 200000, kind)
    _, rc, _, _ = solvers("lean", solver, PL, PR)
    _, full_rc, _, _ = solvers("full", solver, PL, PR)
    assert (full_rc != 0).any()
    assert (rc[full_rc != 0] == DEFER).all()


def test_side_flux_without_density_is_not_a_number(solvers):
    """As from the conserved state, whose enthalpy per mass is infinite there: the predicted
    state's inversion then counts the failure. With a density the two agree to round-off."""
    PL, _ = cold_or_empty(np.random.default_rng(3), 100, "empty")
    F, G = solvers.side_flux(PL)
    assert np.isnan(G[:, 1:5]).all() and np.isnan(F[:, 1:5]).all()
    PL, _ = random_interfaces(np.random.default_rng(3), 20000, 0.1, 1.5, 1.0)
    F, G = solvers.side_flux(PL)
    assert (np.abs(F - G).max(axis=1) <= 1e-13 * np.abs(G).max(axis=1)).all()


@pytest.mark.parametrize("theta", [1.0, 1.5, 2.0])
def test_plm_with_infinities_and_not_a_number(solvers, oracle_lib, theta):
    """The limited state of every triple of ordinary, infinite and not-a-number values is the
    oracle's (equal as numbers or both not a number; with an infinite centre both are infinite or
    not a number, which no solver takes); the form for sweeps that hand such states on gives
    the same or, where one of the three is not finite, not a number. FP32 likewise, by the same
    values (all exact there)."""
    x = [-np.inf, -2.0, -1.0, -0.25, 0.0, 0.5, 1.0, 2.0, np.inf, np.nan]
    V = np.array(np.meshgrid(x, x, x, indexing="ij")).reshape(3, -1).T
    V6 = np.zeros((len(V), 6))
    V6[:, 1:4] = V
    # the oracle takes 6 values v[-2..3]; PLM uses v[-1..1]
    ref = oracle_lib.reconstruct(V6, "PLM_C2R", theta=theta)
    finite = np.isfinite(V).all(axis=1)
    for got, hand_on in zip(*[iter(solvers.plm_ahead(V, theta))] * 2):
        some = ~np.isinf(V[:, 1])
        assert np.array_equal(got[some].astype(float), ref[some], equal_nan=True)
        assert not np.isfinite(got[~some]).any() and not np.isfinite(ref[~some]).any()
        assert np.array_equal(hand_on[finite].astype(float), ref[finite])
        assert (np.isnan(hand_on) | (hand_on.astype(float) == ref)).all()
        # a value that is not a number never goes unseen
        assert np.isnan(hand_on[np.isnan(V).any(axis=1)]).all()


@pytest.mark.parametrize("scale", [1e-8, 1.0, 1e8])
def test_lean_weno5(solvers, scale):
    """The paired finite-volume states and the finite-difference fluxes against the general
    reconstruction, smooth and rough values, constant ones exactly: 4e-14 of the largest value
    (some 50 operations of 2e-16 each, counted four times for the weights, which are fourth
    powers)."""
    rng = np.random.default_rng(5)
    V = rng.uniform(-1, 1, (30000, 6))
    x = np.arange(6) - 2.5
    for k in range(10000):
        V[k] = np.polyval(rng.uniform(-1, 1, 5) * [1e-3, 1e-2, 0.05, 0.2, 1.0], x)
    V[:100] = V[:100, :1]
    V *= scale
    F, G = solvers.weno5(V)
    assert (np.abs(F - G) <= 4e-14 * np.abs(V).max(axis=1, keepdims=True)).all()
    assert np.array_equal(F[:100], np.repeat(V[:100, :1], 4, axis=1))
    assert np.isnan(solvers.weno5(np.where(np.arange(6) == 3, np.nan, V[:1]))[0][:, :3]).all()
