"""The FP64 sweeps where their common path branches, against the oracle: both fast waves on
one side of the interface (the flux of that side, in either direction), the reconstruction
methods it dispatches on, and grids whose sweeps end inside a block.

Tolerances: error counts identical, HLLD counts within 2. The common path takes the
reference's formulas in another order, so it agrees to round-off; at these flow speeds
(W > 2) round-off alone moves the reference's quartic roots, so MaxLambda and the states are
held to the plain form's tolerances (1e-12; 1e-10 in L1, 1e-7 at any zone) or, where that is
more, to 4x of how far the oracle's own run moves under 1-ulp noise on the initial state.
"""
import numpy as np
import pytest

from oracle.oracle import Setup, synchronize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extrap,IS,flow,N,riemann", [
    ("weno5", "js96", (0.95, 0.0, 0.0), (13, 18, 11), "hlld"),
    ("weno5", "js96", (0.0, -0.9, 0.3), (9, 14, 22), "hlld"),
    ("weno5", "sz10", (0.2, 0.1, 0.93), (12, 10, 19), "hlld"),
    ("plm", "js96", (-0.93, 0.2, 0.0), (17, 8, 15), "hlld"),
    ("pcm", "js96", (0.0, 0.0, -0.95), (10, 11, 33), "hlld"),
    ("plm", "js96", (0.0, 0.93, 0.1), (11, 9, 13), "hll"),
    ("weno5", "js96", (-0.9, 0.0, 0.3), (14, 9, 16), "hllc"),
])
def test_supersonic_sweeps(gpu, oracle_lib, extrap, IS, flow, N, riemann):
    rng = np.random.default_rng(sum(N))
    x = [2 * np.pi * (np.arange(n) + 0.5) / n for n in N]
    X, Y, Z = np.meshgrid(*x, indexing="ij")
    P = np.empty(tuple(n + 6 for n in N) + (8,))
    it = (slice(3, -3),) * 3
    wave = [np.sin(X + p) * np.cos(Y + q) + np.sin(Z + r) for p, q, r in rng.uniform(0, 6, (8, 3))]
    P[it + (0,)] = 1.0 + 0.2 * wave[0]
    P[it + (1,)] = 0.2 * (1.0 + 0.2 * wave[1])
    for d in range(3):
        P[it + (2 + d,)] = flow[d] + 0.01 * wave[2 + d]
        P[it + (5 + d,)] = (0.2, 0.15, 0.25)[d] + 0.02 * wave[5 + d]
    P = synchronize(P, 3)
    s = Setup(N=N, extrap=extrap, IS=IS, riemann=riemann, advance="rk2")

    def march(P0):
        so = oracle_lib.solver(s)
        Po, dt, out = P0.copy(), 0.0, []
        for _ in range(3):
            eo, sto = so.advance(Po, dt)
            out.append((eo, sto.hlld_success, sto.max_lambda, dt))
            dt = so.get_timestep(0.4)
        return Po, out

    Po, ref = march(P)
    lam_tol = np.full(3, 1e-12)
    L1_tol, max_tol = np.full(8, 1e-10), np.full(8, 1e-7)
    L1 = lambda A: np.abs(A - Po).sum(axis=(0, 1, 2)) / np.abs(Po).sum(axis=(0, 1, 2))  # noqa: E731
    worst = lambda A: np.abs(A - Po).max(axis=(0, 1, 2)) / np.abs(Po).max(axis=(0, 1, 2))  # noqa: E731
    for _ in range(8):
        Pn, noisy = march(P * (1 + 2.3e-16 * rng.choice([-1, 0, 1], size=P.shape)))
        lam_tol = np.maximum(lam_tol, [4 * abs(a[2] - b[2]) / b[2] for a, b in zip(noisy, ref)])
        L1_tol, max_tol = np.maximum(L1_tol, 4 * L1(Pn)), np.maximum(max_tol, 4 * worst(Pn))

    ctx = gpu.Context(gpu.make_config(N=N, extrap=extrap, IS=IS, riemann=riemann, advance="rk2"))
    ctx.upload(P)
    for (eo, ok, lam, dt), tol in zip(ref, lam_tol):
        eg, stg = ctx.advance(dt)
        assert eo == eg == 0
        assert abs(stg.max_lambda - lam) <= tol * lam
        assert abs(stg.hlld_success - ok) <= 2
    Pg = ctx.download()
    assert (L1(Pg) <= L1_tol).all()
    assert (worst(Pg) <= max_tol).all()


@pytest.mark.parametrize("N,Ng,extrap,riemann,precision", [
    ((3, 3, 3), 3, "weno5", "hlld", "fp64"),
    ((3, 3, 3), 3, "weno5", "hlld", "mixed"),
    ((4, 3, 67), 2, "plm", "hlld", "fp64"),
    ((5, 40, 4), 3, "plm", "hllc", "fp64"),
    ((33, 3, 5), 3, "weno5", "hlld", "mixed"),
])
def test_smallest_grids(gpu, oracle_lib, N, Ng, extrap, riemann, precision):
    """The three sweeps of a stage share one launch, each with its own range of blocks: grids
    whose ranges are empty, shorter than a block, or end inside a block or a tile column.
    Plain-form tolerances (mixed: 1e-6 in L1, its bound against FP64)."""
    rng = np.random.default_rng(sum(N) + Ng)
    P = np.empty(tuple(n + 2 * Ng for n in N) + (8,))
    it = (slice(Ng, -Ng),) * 3
    P[it] = [1.0, 0.6, 0.1, -0.05, 0.08, 0.3, 0.2, 0.4]
    P[it] *= 1.0 + 0.02 * rng.uniform(-1, 1, tuple(N) + (8,))
    P = synchronize(P, Ng)
    so = oracle_lib.solver(Setup(N=N, Ng=Ng, extrap=extrap, riemann=riemann, advance="rk3"))
    ctx = gpu.Context(gpu.make_config(N=N, Ng=Ng, extrap=extrap, riemann=riemann, advance="rk3", precision=precision))
    ctx.upload(P)
    Po, dt = P.copy(), 0.1 / max(N)
    for _ in range(2):
        eo, sto = so.advance(Po, dt)
        eg, stg = ctx.advance(dt)
        assert eo == eg == 0
        tol = 1e-12 if precision == "fp64" else 1e-5
        assert abs(stg.max_lambda - sto.max_lambda) <= tol * sto.max_lambda
    Pg = ctx.download()
    L1 = np.abs(Pg - Po).sum(axis=(0, 1, 2)) / np.abs(Po).sum(axis=(0, 1, 2))
    assert L1.max() < (1e-10 if precision == "fp64" else 1e-6)


@pytest.mark.parametrize("riemann", ["hll", "hlld"])
def test_single_zone(gpu, riemann):
    """One zone with one ghost zone a side: no interface along x at all (an empty range of
    blocks), and a uniform state, which no step changes beyond round-off."""
    P = np.tile(np.array([1.0, 0.6, 0.1, -0.05, 0.08, 0.3, 0.2, 0.4]), (3, 3, 3, 1))
    ctx = gpu.Context(gpu.make_config(N=(1, 1, 1), Ng=1, extrap="pcm", riemann=riemann, advance="rk3"))
    ctx.upload(P)
    for _ in range(2):
        assert ctx.advance(0.1)[0] == 0
    assert np.abs(ctx.download() - P).max() < 1e-14


@pytest.mark.parametrize("n", [8, 38])
def test_full_solver_queue(gpu, oracle_lib, n):
    """Rough states, whose interfaces leave the common path in number: few enough that the full
    solver gives each 16 lanes (n = 8), and more than 4096 in a launch, one lane each (n = 38).
    The HLLD counts and the state after one small step against the oracle, held to 4x its own
    spread under 1-ulp noise (the attempt ladder flips there) or the plain tolerances."""
    rng = np.random.default_rng(n)
    N = (n, n, n)
    P = np.empty((n + 6,) * 3 + (8,))
    it = (slice(3, -3),) * 3
    r = rng.uniform(-1, 1, N + (8,))
    P[it + (0,)] = np.exp(1.5 * r[..., 0])
    P[it + (1,)] = np.exp(2.0 * r[..., 1])
    P[it + (slice(2, 5),)] = 0.5 * r[..., 2:5]
    P[it + (slice(5, 8),)] = 2.0 * r[..., 5:8]
    P = synchronize(P, 3)
    kw = dict(N=N, extrap="plm", riemann="hlld", advance="single")

    def step(P0):
        so = oracle_lib.solver(Setup(**kw))
        Q = P0.copy()
        e, st = so.advance(Q, 1e-3 / n)
        return e, st.hlld_success, st.hlld_failure, Q

    e0, ok0, fail0, Q0 = step(P)
    L1 = lambda Q: np.abs(Q - Q0).sum(axis=(0, 1, 2)) / np.abs(Q0).sum(axis=(0, 1, 2))  # noqa: E731
    ok_tol, tol = 2.0, np.full(8, 1e-10)
    for _ in range(8):
        e, ok, fail, Q = step(P * (1 + 2.3e-16 * rng.choice([-1, 0, 1], size=P.shape)))
        ok_tol = max(ok_tol, 4 * abs(ok - ok0))
        tol = np.maximum(tol, 4 * L1(Q))
    assert e0 == 0 and fail0 > (100 if n == 8 else 6000)
    ctx = gpu.Context(gpu.make_config(**kw))
    ctx.upload(P)
    eg, st = ctx.advance(1e-3 / n)
    assert eg == 0
    assert (st.fp64_redo <= 4096) == (n == 8)
    assert st.hlld_success + st.hlld_failure == ok0 + fail0
    assert abs(st.hlld_success - ok0) <= ok_tol
    assert (L1(ctx.download()) <= tol).all()


@pytest.mark.parametrize("seed", [412, 436, 409])
def test_weak_normal_field(gpu, oracle_lib, seed):
    """Interfaces whose normal field nearly vanishes, where the p* solve ends by its own
    shortcuts: whether HLLD is accepted there, and at which root, is the reference's. The
    first two states hold an interface that reaches the last Newton step. Tolerances: HLLD
    failures within 2, states within the plain form's 1e-7 at any zone (a flipped decision
    moves them by 2e-5 and more; 1-ulp noise moves the oracle's by 3e-14 here)."""
    N, dx = (20, 16, 24), 1.0 / 24
    x1 = tuple(n * dx for n in N)
    P = gpu.init_turbulence(N, Ng=3, seed=seed, v_rms=0.3, v_kmax=4.0, four_velocity=False, B0=(0.0, 0.0, 1.0),
                            dB_rms=0.3, A_kmax=3.0)
    so = oracle_lib.solver(Setup(N=N, x1=x1, extrap="plm", riemann="hlld", advance="rk2"))
    ctx = gpu.Context(gpu.make_config(N=N, x1=x1, extrap="plm", riemann="hlld", advance="rk2"))
    ctx.upload(P)
    Po, dt = P.copy(), 0.4 * dx
    for _ in range(8):
        eo, sto = so.advance(Po, dt)
        eg, stg = ctx.advance(dt)
        assert eo == eg == 0
        assert abs(stg.hlld_failure - sto.hlld_failure) <= 2
        dt = so.get_timestep(0.4)
    d = np.abs(ctx.download() - Po).max(axis=(0, 1, 2)) / np.abs(Po).max(axis=(0, 1, 2))
    assert (d <= 1e-7).all()


@pytest.mark.parametrize("riemann", ["hll", "hllc"])
def test_retry_queue_hll(gpu, oracle_lib, riemann):
    """A zone next to the light cone, whose neighbours' reconstructed states pass it: those
    interfaces go to the full solver, which retries with the zone-centred states, in the HLL and
    HLLC sweeps too. Counts as the oracle's, the state as in test_supersonic_sweeps (one small
    step, so nothing has time to grow)."""
    N = (9, 8, 12)
    rng = np.random.default_rng(3)
    P = np.empty(tuple(n + 6 for n in N) + (8,))
    it = (slice(3, -3),) * 3
    P[it] = [1.0, 1.0, 0.5, 0.1, 0.0, 0.2, 0.3, 0.1]
    P[it + (slice(2, 5),)] += 0.3 * rng.uniform(-1, 1, N + (3,))
    P[7, 6, 8, 2:5] = (0.99, 0.1, 0.05)
    P[6, 6, 8, 2:5] = (0.8, 0.1, 0.05)
    P[8, 6, 8, 2:5] = (0.9, 0.4, 0.05)
    P = synchronize(P, 3)
    kw = dict(N=N, extrap="weno5", riemann=riemann, advance="single")
    so = oracle_lib.solver(Setup(**kw))
    Po = P.copy()
    eo, sto = so.advance(Po, 1e-4)
    ctx = gpu.Context(gpu.make_config(**kw))
    ctx.upload(P)
    eg, stg = ctx.advance(1e-4)
    assert eo == eg == 0 and sto.riemann_retries > 0
    assert stg.riemann_retries == sto.riemann_retries == stg.fp64_redo
    assert stg.riemann_failures == sto.riemann_failures
    Pg = ctx.download()
    assert (np.abs(Pg - Po).sum(axis=(0, 1, 2)) / np.abs(Po).sum(axis=(0, 1, 2))).max() < 1e-10


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("N,Ng,IS", [((3, 5, 4), 3, "js96"), ((58, 4, 59), 3, "js96"), ((6, 60, 118), 4, "sz10"),
                                     ((65, 7, 5), 3, "b08")])
def test_weno_split_tiles(gpu, oracle_lib, N, Ng, IS, precision):
    """The component-wise weno-split kernel at the edges of its tiles: one tile of interfaces
    along an axis (up to 59), one more, two full ones, lines that fill no block, more ghost zones
    than the stencil needs, the other smoothness indicators. Two steps against the oracle,
    plain-form tolerances (mixed: L1 1e-6, its bound against FP64)."""
    rng = np.random.default_rng(sum(N))
    P = np.empty(tuple(n + 2 * Ng for n in N) + (8,))
    it = (slice(Ng, -Ng),) * 3
    P[it] = [1.0, 0.6, 0.1, -0.05, 0.08, 0.3, 0.2, 0.4]
    P[it] *= 1.0 + 0.02 * rng.uniform(-1, 1, tuple(N) + (8,))
    P = synchronize(P, Ng)
    kw = dict(N=N, Ng=Ng, godunov="weno-split", extrap="weno5", IS=IS, advance="rk2")
    so = oracle_lib.solver(Setup(**kw))
    ctx = gpu.Context(gpu.make_config(precision=precision, **kw))
    ctx.upload(P)
    Po, dt = P.copy(), 0.1 / max(N)
    for _ in range(2):
        eo, sto = so.advance(Po, dt)
        eg, stg = ctx.advance(dt)
        assert eo == eg == 0
        assert abs(stg.max_lambda - sto.max_lambda) <= (1e-12 if precision == "fp64" else 1e-5) * sto.max_lambda
    Pg = ctx.download()
    L1 = np.abs(Pg - Po).sum(axis=(0, 1, 2)) / np.abs(Po).sum(axis=(0, 1, 2))
    assert L1.max() < (1e-10 if precision == "fp64" else 1e-6)


@pytest.mark.parametrize("N,B,v", [
    ((7, 5, 6), (0.0, 0.0, 0.0), 0.3),        # no field: every spectrum has a cluster
    ((5, 9, 4), (0.9, 0.0, 0.0), 0.2),        # no normal field along y and z
    ((11, 4, 5), (0.5, 0.3, -0.4), 0.0),      # at rest: lam = 0 and vn coincide
    ((4, 6, 9), (0.5, 0.3, -0.4), 0.3),       # simple spectra
])
def test_weno_split_characteristic_queue(gpu, oracle_lib, N, B, v):
    """The characteristic sweep where its short projection does not apply (clusters of
    eigenvalues, left to the general eigensystem) and where it does, against the oracle. The
    basis of a cluster's eigenspace follows round-off, so the state is held to 4x the oracle's
    own spread under 1-ulp noise, or to 1e-10 in L1."""
    rng = np.random.default_rng(sum(N))
    P = np.empty(tuple(n + 6 for n in N) + (8,))
    it = (slice(3, -3),) * 3
    P[it] = [1.0, 0.6, 0.0, 0.0, 0.0, *B]
    P[it + (slice(0, 2),)] *= 1.0 + 0.05 * rng.uniform(-1, 1, N + (2,))
    P[it + (slice(2, 5),)] += v * rng.uniform(-1, 1, N + (3,))
    P = synchronize(P, 3)
    kw = dict(N=N, godunov="weno-split", eigen="rmhd", extrap="weno5", advance="rk2")

    def march(P0):
        so = oracle_lib.solver(Setup(**kw))
        Q = P0.copy()
        errors = [so.advance(Q, 0.05 / max(N))[0] for _ in range(2)]
        return errors, Q

    e0, Q0 = march(P)
    L1 = lambda Q: np.abs(Q - Q0).sum(axis=(0, 1, 2)) / np.maximum(np.abs(Q0).sum(axis=(0, 1, 2)), 1e-3)  # noqa: E731
    tol = np.full(8, 1e-10)
    for _ in range(8):
        _, Qn = march(P * (1 + 2.3e-16 * rng.choice([-1, 0, 1], size=P.shape)))
        tol = np.maximum(tol, 4 * L1(Qn))
    ctx = gpu.Context(gpu.make_config(**kw))
    ctx.upload(P)
    assert [ctx.advance(0.05 / max(N))[0] for _ in range(2)] == e0 == [0, 0]
    assert (L1(ctx.download()) <= tol).all()


@pytest.mark.parametrize("N,B,godunov,extrap", [
    ((20, 24, 18), 1e-6, "plm-split", "weno5"),   # every interface leaves the lean path
    ((33, 17, 20), 1e-5, "plm-split", "plm"),     # about half
    ((18, 20, 25), 1e-6, "plm-muscl", "plm"),
    ((17, 24, 19), 20.0, "plm-split", "weno5"),   # a dominating field: some need the whole ladder
])
def test_long_queue(gpu, oracle_lib, N, B, godunov, extrap):
    """A weak or a dominating field, where most interfaces go through the bulk kernel, against
    the oracle: error counts, and HLLD successes and states within the plain tolerances or 4x
    the oracle's own spread under 1-ulp noise."""
    P = gpu.init_turbulence(N, Ng=3, seed=7, v_rms=0.3, v_kmax=4.0, four_velocity=False, B0=(0.3 * B, 0.2 * B, B),
                            dB_rms=0.3 * B, A_kmax=3.0)
    kw = dict(N=N, x1=tuple(n / max(N) for n in N), extrap=extrap, riemann="hlld", advance="rk2", godunov=godunov)
    dt = 0.1 / max(N)

    def march(P0):
        so, Q, out = oracle_lib.solver(Setup(**kw)), P0.copy(), []
        for _ in range(1 if B > 1 else 2):       # at B = 20 the reference's second step fails
            e, st = so.advance(Q, dt)
            out.append((e, st.hlld_success, st.hlld_failure))
        return Q, out

    Q0, ref = march(P)
    rng = np.random.default_rng(1)
    L1 = lambda Q: np.abs(Q - Q0).sum(axis=(0, 1, 2)) / np.abs(Q0).sum(axis=(0, 1, 2))  # noqa: E731
    tol, ok_tol = np.full(8, 1e-10), np.full(len(ref), 2.0)
    for _ in range(8):
        Q, out = march(P * (1 + 2.3e-16 * rng.choice([-1, 0, 1], size=P.shape)))
        tol = np.maximum(tol, 4 * L1(Q))
        ok_tol = np.maximum(ok_tol, [4 * abs(a[1] - b[1]) for a, b in zip(out, ref)])
    ctx = gpu.Context(gpu.make_config(**kw))
    ctx.upload(P)
    for (e0, ok0, fail0), ok_t in zip(ref, ok_tol):
        e, st = ctx.advance(dt)
        assert e == e0 == 0
        assert st.fp64_redo > 2 * 4096
        assert st.hlld_success + st.hlld_failure == ok0 + fail0
        assert abs(st.hlld_success - ok0) <= ok_t
    assert (L1(ctx.download()) <= tol).all()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("B0,dB,share", [
    ((0.0, 0.0, 0.0), 0.0, (1.0, 1.0)),        # no field: every spectrum has a cluster
    ((1e-4, 2e-4, 1e-4), 3e-5, (1.0, 1.0)),    # the slow speeds within 1e-7 of the Alfven ones
    ((0.5, 0.6, 0.7), 0.3, (0.0, 0.05)),       # simple spectra but for a few
])
def test_characteristic_interfaces_handed_on(gpu, B0, dB, share, precision):
    """Which interfaces of the characteristic sweep go to the general eigensystem: all of them
    with clusters everywhere, next to none otherwise (fp64_redo; one stage, so once per interface
    of the three sweeps, whose transverse lines include the ghosts)."""
    N = (19, 14, 22)
    P = gpu.init_turbulence(N, Ng=3, seed=3, v_rms=0.3, v_kmax=4.0, four_velocity=False, B0=B0, dB_rms=dB, A_kmax=3.0)
    ctx = gpu.Context(gpu.make_config(N=N, godunov="weno-split", eigen="rmhd", extrap="weno5", advance="single",
                                      precision=precision))
    ctx.upload(P)
    e, st = ctx.advance(1e-3)
    n = [k + 6 for k in N]
    total = (N[0] + 1) * n[1] * n[2] + n[0] * (N[1] + 1) * n[2] + n[0] * n[1] * (N[2] + 1)
    assert e == 0 and st.fp64_redo_overflow == 0
    assert share[0] * total <= st.fp64_redo <= share[1] * total


@pytest.mark.parametrize("N,extrap,riemann", [((17, 12, 26), "plm", "hllc"), ((9, 22, 13), "weno5", "hllc"),
                                              ((12, 31, 10), "weno5", "hll")])
def test_mixed_full_solver_sweeps(gpu, oracle_lib, N, extrap, riemann):
    """The mixed form's HLL and HLLC sweeps (three axes in one launch, the full FP32 solver) on
    grids whose axes differ, against the oracle: the bounds of the mixed form's other steps, L1
    1e-5 and the fastest speed to 1e-4. The field is oblique: with a normal field that passes
    zero HLLC multiplies round-off, and the oracle's own speeds move by 5e-5 under FP32
    rounding of the state (here by 4e-8)."""
    P0 = gpu.init_turbulence(N, v_rms=0.3, v_kmax=3.0, four_velocity=True, B0=(0.6, 0.6, 0.6), dB_rms=0.2,
                             A_kmax=2.0, seed=11)
    kw = dict(N=N, x1=tuple(n / max(N) for n in N), extrap=extrap, riemann=riemann, advance="rk2")
    so = oracle_lib.solver(Setup(**kw))
    ctx = gpu.Context(gpu.make_config(precision="mixed", **kw))
    ctx.upload(P0)
    Po, dt = P0.copy(), 0.1 / max(N)
    for _ in range(3):
        eo, sto = so.advance(Po, dt)
        eg, stg = ctx.advance(dt)
        assert eo == eg == 0
        assert abs(stg.max_lambda - sto.max_lambda) <= 1e-4 * sto.max_lambda
    it = (slice(3, -3),) * 3
    a, b = ctx.download()[it], Po[it]
    assert (np.abs(a - b).sum(axis=(0, 1, 2)) <= 1e-5 * np.abs(b).sum(axis=(0, 1, 2))).all()
