"""The chip-resident time loop (dn_resident.*) against the sweeps and the FP32
oracle: one grid per thread shape (1x1, 1x2, 1x4, 2x4, 3x4 cells per thread)
with ragged last tiles, every operator length, points on tile edges, runs
longer than one launch.  A context whose caller chose a sweep shape takes the
sweeps; all other runs here fit the loop.  The arithmetic is the same term by
term, so everything compares bit for bit."""
import numpy as np
import pytest

import dnhip
import orc
import synth
from cases import make_case

pytestmark = pytest.mark.gpu


def context(case, sweeps):
    p, m, src, sig, rec = case
    g = dnhip.Context(p)
    if p.physics in (3, 4):
        g.set_model_aniso(*synth.anisotropic_model(p.nx, p.ny, p.dh, 5, sigma=3.0,
                                                   tilt=20.0 if p.physics == 4 else None))
    else:
        g.set_model(m["vp"], m["vs"], m["rho"], m["taus"], m["taup"])
    if sweeps:
        g.set_tile(64, 4, 1, 1)
    g.set_sources(src, sig)
    g.set_receivers(rec)
    return g


def state(g, p):
    out = [g.seismogram(k) for k in range(5)] + [g.field(f) for f in range(7)] + [g.psi(k) for k in range(9)]
    return out + [g.memvar(w, l + 1) for w in range(3) for l in range(p.L)]


def check_forward(case, steps=0):
    a, b = context(case, False), context(case, True)
    print(f"resident run {case[0].nx}x{case[0].ny} order {case[0].fdorder}", flush=True)
    a.forward(steps)
    b.forward(steps)
    assert np.abs(a.field(dnhip.F_VX)).max() > 0
    for k, (x, y) in enumerate(zip(state(a, case[0]), state(b, case[0]))):
        np.testing.assert_array_equal(x, y, err_msg=f"output {k}")
    return a


# grids: one tile; ragged tiles of 1x1, 1x2, 1x4, 2x4 and 3x4 cells per thread
GRIDS = [(29, 21), (131, 77), (611, 303), (1003, 401), (1201, 601), (1502, 602), (1997, 598)]


@pytest.mark.parametrize("free_surf", [0, 1])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_forward_equals_sweeps_on_every_thread_shape(nx, ny, free_surf):
    fw = 5 if ny < 40 else 10
    check_forward(make_case(nx=nx, ny=ny, nt=60, fdorder=8, fw=fw, free_surf=free_surf, seismo=4, homogeneous=True,
                            nrec=max(3, nx // 2 - 4)))


@pytest.mark.parametrize("fdorder", [2, 4, 6, 8, 10, 12])
def test_forward_equals_oracle_for_every_order(fdorder):
    case = make_case(nx=173, ny=61, nt=150, fdorder=fdorder, fw=7, seismo=4, free_surf=fdorder // 2 % 2)
    g = check_forward(case)
    p, m, src, sig, rec = case
    o = orc.Oracle(p, m["vp"], m["vs"], m["rho"], prec="f32")
    o.set_sources(src, sig)
    o.set_receivers(rec)
    o.forward()
    for k in range(5):
        np.testing.assert_array_equal(g.seismogram(k), o.seismogram(k))


@pytest.mark.parametrize("stype", [1, 2, 3, 4])
def test_points_on_tile_edges(stype):
    """Sources and receivers in the last and first cells of tiles (32 columns
    and up to 32 rows), the grid's corners among them, several per cell."""
    case = make_case(nx=140, ny=90, nt=120, fw=10, seismo=4, stype=stype)
    p, m, src, sig, rec = case
    src = np.repeat(src, 3, 1)
    src[0] = [32, 33, 33]
    src[1] = [2, 40, 40]
    sig = np.repeat(sig, 3, 0) * np.array([[1.0], [0.5], [-0.25]], np.float32)
    xs = [1, 31, 32, 33, 64, 65, 96, 97, 139, 140]
    ys = [1, 2, 3, 4, 5, 6, 9, 44, 89, 90]
    rec = np.array([[x for x in xs for _ in ys], [y for _ in xs for y in ys]], np.int32)
    check_forward((p, m, src, sig, rec))


def test_surface_source_and_long_runs():
    """An explosive source in the surface row (applied before the surface
    condition: the sweeps take it), and a run of several launches."""
    case = make_case(nx=90, ny=60, nt=100, src_xz=(450.0, 10.0))
    check_forward(case)
    check_forward(make_case(nx=90, ny=60, nt=4500, fw=10))
    check_forward(make_case(nx=90, ny=60, nt=400, fw=10), steps=33)


def gradient(case, sweeps):
    g = context(case, sweeps)
    print(f"resident gradient physics {case[0].physics} {case[0].nx}x{case[0].ny} sweeps {sweeps}", flush=True)
    g.forward()
    seis = [g.seismogram(k) for k in range(5)]
    rng = np.random.default_rng(3)
    adj = [(rng.standard_normal((g.ntr, case[0].nt)) * 1e-6).astype(np.float32) for _ in range(3)]
    g.set_adjoint_sources(*adj)
    g.adjoint()
    out = seis + [g.gradient(k) for k in range(3)] + [g.field(f) for f in range(7)] + [g.psi(k) for k in range(9)]
    if case[0].physics not in (3, 4):
        g.assemble()
        out += [g.gradient(k) for k in range(3, 6)]
    g.close()
    return out


@pytest.mark.parametrize("nx,ny,dtinv", [(131, 77, 1), (256, 120, 3), (612, 302, 2), (1201, 601, 4), (1997, 598, 3)])
def test_gradient_equals_sweeps(nx, ny, dtinv):
    """Stored snapshots and the adjoint run with its correlations, odd NX and
    the unaligned snapshot rows it brings among them."""
    case = make_case(nx=nx, ny=ny, nt=70, fw=10, mode=1, dtinv=dtinv, homogeneous=True)
    a, b = gradient(case, False), gradient(case, True)
    assert np.abs(a[5]).max() > 0
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("quelltypb", [1, 2, 3, 4, 7])
def test_adjoint_source_types(quelltypb):
    case = make_case(nx=140, ny=90, nt=80, fw=10, mode=1, dtinv=2, quelltypb=quelltypb, seismo=4)
    for x, y in zip(gradient(case, False), gradient(case, True)):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("nx,ny,fdorder,free_surf", [(29, 21, 4, 1), (140, 90, 2, 0), (173, 61, 12, 1),
                                                     (811, 303, 8, 1), (1201, 601, 8, 0), (1997, 598, 8, 1)])
@pytest.mark.parametrize("physics", [2, 3, 4, 5])
def test_other_physics_equal_sweeps(physics, nx, ny, fdorder, free_surf):
    """Acoustic, VTI, TTI and SH runs, forward with snapshots and adjoint."""
    case = make_case(nx=nx, ny=ny, nt=60, fdorder=fdorder, fw=5 if ny < 40 else 10, mode=1, dtinv=2, safety=0.5,
                     free_surf=free_surf, seismo={2: 2, 5: 1}.get(physics, 4), homogeneous=True)
    case[0].physics = physics
    a, b = gradient(case, False), gradient(case, True)
    assert max(np.abs(x).max() for x in a[5:8]) > 0
    for k, (x, y) in enumerate(zip(a, b)):
        np.testing.assert_array_equal(x, y, err_msg=f"output {k}")


@pytest.mark.parametrize("L", [1, 2, 3])
@pytest.mark.parametrize("nx,ny,fdorder,free_surf", [(140, 90, 8, 1), (331, 303, 12, 0), (1003, 401, 8, 1),
                                                     (1201, 601, 4, 1), (1997, 598, 8, 1)])
def test_viscoelastic_equals_sweeps(L, nx, ny, fdorder, free_surf):
    """Forward runs with their memory variables, and gradients."""
    kw = dict(nx=nx, ny=ny, nt=60, fdorder=fdorder, fw=10, L=L, free_surf=free_surf, seismo=4, homogeneous=True)
    check_forward(make_case(**kw))
    case = make_case(mode=1, dtinv=2, **kw)
    for k, (x, y) in enumerate(zip(gradient(case, False), gradient(case, True))):
        np.testing.assert_array_equal(x, y, err_msg=f"output {k}")


def test_concurrent_contexts():
    """More runs at once than the CUs take: those without room take the
    sweeps, and every result is the run's own."""
    import threading
    cases = [make_case(nx=400 + 20 * k, ny=200, nt=150, fw=10, seed=k + 1) for k in range(4)]
    want = []
    for c in cases:
        g = context(c, True)
        g.forward()
        want.append(g.seismogram(0))
    ctx = [context(c, False) for c in cases]
    bad = []

    def work(k):
        for _ in range(3):
            ctx[k].forward()
            if not np.array_equal(ctx[k].seismogram(0), want[k]):
                bad.append(k)

    print("concurrent resident runs", flush=True)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("steps", [[200], [40, 3, 17, 5, 9, 200]])
@pytest.mark.parametrize("large", [False, True])
def test_engine_rounds_equal_sweeps(steps, large):
    """Shots of several orders, sizes, lengths and relaxation counts together
    (the loop's rounds, large: and a grid for the sweeps, which the small
    rounds join), runs of steps that move them between the loop and the
    sweeps, and a shot that joins on the way."""
    sizes = [(131, 77, 90, 8, 0), (611, 303, 70, 8, 0), (1003, 401, 50, 8, 0), (29, 21, 130, 8, 0), (733, 290, 80, 4, 0),
             (260, 120, 60, 4, 1), (320, 200, 75, 8, 2), (210, 90, 40, 12, 3)]
    if large:
        sizes += [(1301, 801, 40, 8, 0), (2600, 900, 30, 8, 0)]
    cases = [make_case(nx=nx, ny=ny, nt=nt, fdorder=o, L=L, fw=5 if ny < 40 else 10, seismo=4, homogeneous=True,
                       nrec=nx // 3, seed=k + 1) for k, (nx, ny, nt, o, L) in enumerate(sizes)]
    eng = dnhip.Engine()
    shots = [context(c, False) for c in cases]
    for g in shots[1:]:
        eng.attach(g)
    print("rounds of chip-resident shots", flush=True)
    for k, n in enumerate(steps):
        eng.step(n)
        if k == 0:
            eng.attach(shots[0])
    eng.run()
    for case, g in zip(cases, shots):
        assert eng.status(g) == 0
        ref = context(case, True)
        ref.forward()
        assert np.abs(ref.field(dnhip.F_VX)).max() > 0
        for k, (x, y) in enumerate(zip(state(g, case[0]), state(ref, case[0]))):
            np.testing.assert_array_equal(x, y, err_msg=f"{case[0].nx}x{case[0].ny} output {k}")


def test_engine_gradient_rounds_equal_sweeps():
    """Forward and adjoint phases of two grids in the engine's rounds."""
    cases = [make_case(nx=nx, ny=ny, nt=120, fw=10, mode=1, dtinv=2, fc=15.0, nrec=nx // 4, seed=nx)
             for nx, ny in [(333, 150), (905, 411)]]
    eng = dnhip.Engine()
    for chunk in (16, 200):
        shots = [context(c, False) for c in cases]
        for g in shots:
            eng.attach(g, 0)
        eng.run(chunk)
        for g in shots:
            zero = np.zeros_like(g.seismogram(0))
            g.residuals(zero, zero, None, 1)
            eng.attach(g, 1)
        print("gradient rounds", flush=True)
        eng.run(chunk)
        for case, g in zip(cases, shots):
            ref = context(case, True)
            ref.forward()
            zero = np.zeros_like(ref.seismogram(0))
            ref.residuals(zero, zero, None, 1)
            ref.adjoint()
            g.assemble()
            ref.assemble()
            for w in range(6):
                np.testing.assert_array_equal(g.gradient(w), ref.gradient(w), err_msg=f"{case[0].nx} gradient {w}")


def test_engine_parts_equal_single_shots():
    """Three grids that together exceed the last-level cache: the engine runs
    them in parts, each through a whole run of steps, with and without a
    graph, while a small shot ends between them."""
    cases = [make_case(nx=nx, ny=ny, nt=nt, fdorder=8, fw=10, seismo=1, homogeneous=True, nrec=nx // 9, seed=k + 1)
             for k, (nx, ny, nt) in enumerate([(2600, 900, 26), (2400, 1000, 37), (2500, 950, 30), (60, 50, 21)])]
    print("parts of the engine's sweeps", flush=True)
    shots = [context(c, True) for c in cases]
    for g in shots:
        g.forward()
    want = [(g.seismogram(0), g.field(dnhip.F_SXX)) for g in shots]
    for graph in (0, 8):
        eng = dnhip.Engine()
        eng.set_graph(graph)
        for g in shots:
            eng.attach(g)
        while eng.step(16) > 0:
            pass
        for g, (s, f) in zip(shots, want):
            assert eng.status(g) == 0
            assert np.abs(f).max() > 0
            np.testing.assert_array_equal(g.seismogram(0), s)
            np.testing.assert_array_equal(g.field(dnhip.F_SXX), f)
