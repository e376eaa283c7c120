"""Which path a run takes, and every compiled kernel of the chip-resident time
loop against the sweeps.  The loop's arithmetic is the sweeps' term by term, so
everything compares bit for bit; dn_get_loop says what ran."""
import numpy as np
import pytest

import dnhip
from cases import make_case
from test_gpu_resident import context, state

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 2), (1, 4), (2, 4), (3, 4)]


def rows(fdorder, physics, L, adjoint):
    """Rows per thread, at most, of the compiled kernels (res_rows)."""
    if L > 0:
        return 1 if L > 2 or adjoint else 2 if L == 2 and fdorder != 8 else 3
    if physics == 4:
        return 3 if fdorder == 8 else (1 if fdorder > 8 else 2) if adjoint else 2 if fdorder > 8 else 3
    return 3 - adjoint if physics in (1, 3) and fdorder > 8 else 3


def small(fdorder, physics, L, free_surf=1):
    # three columns of tiles of every width, several rows of tiles, ragged last ones
    case = make_case(nx=167, ny=83, nt=40, fdorder=fdorder, fw=9, L=L, mode=1, dtinv=3, safety=0.5, homogeneous=True,
                     free_surf=free_surf, seismo={2: 2, 5: 1}.get(physics, 4), nrec=60)
    case[0].physics = physics
    return case


def forward_and_adjoint(g, p):
    """Outputs of both halves, and the paths they took."""
    g.forward()
    out, path = state(g, p), [g.loop()]
    rng = np.random.default_rng(3)
    g.set_adjoint_sources(*[(rng.standard_normal((g.ntr, p.nt)) * 1e-6).astype(np.float32) for _ in range(3)])
    g.adjoint()
    path.append(g.loop())
    return out + [g.gradient(k) for k in range(3)] + state(g, p), path


@pytest.mark.parametrize("fdorder", [2, 4, 6, 8, 10, 12])
@pytest.mark.parametrize("physics,L", [(1, 0), (1, 1), (1, 2), (1, 3), (2, 0), (3, 0), (4, 0), (5, 0)])
def test_every_compiled_shape_equals_the_sweeps(physics, L, fdorder):
    case = small(fdorder, physics, L, free_surf=fdorder // 2 % 2)
    p = case[0]
    g = context(case, True)
    want, path = forward_and_adjoint(g, p)
    assert path == [(0, 0, 0)] * 2
    assert max(np.abs(w).max() for w in want) > 0
    for shape in SHAPES:
        if shape[0] > rows(fdorder, physics, L, 0):
            with pytest.raises(dnhip.DnError):
                g.set_loop(*shape)
            continue
        g.set_loop(*shape)
        print(f"loop physics {physics} L {L} order {fdorder} shape {shape}", flush=True)
        got, path = forward_and_adjoint(g, p)
        assert path == [shape + (0,), (shape if shape[0] <= rows(fdorder, physics, L, 1) else (0, 0)) + (0,)]
        for k, (x, y) in enumerate(zip(got, want)):
            np.testing.assert_array_equal(x, y, err_msg=f"shape {shape} output {k}")


# the library's own choice: grid, order, physics, L, forward shape, adjoint shape
CHOICES = [(131, 77, 8, 1, 0, (1, 1), (1, 1)), (1003, 401, 8, 1, 0, (1, 2), (1, 2)), (1200, 420, 8, 1, 0, (1, 4), (1, 4)),
           (1000, 500, 12, 1, 1, (1, 4), (1, 4)), (1201, 601, 4, 1, 0, (2, 4), (2, 4)), (1237, 431, 12, 1, 1, (2, 4), (0, 0)),
           (1997, 598, 2, 1, 0, (3, 4), (3, 4)), (1701, 550, 10, 1, 0, (2, 4), (2, 4)), (1997, 598, 10, 1, 0, (3, 4), (0, 0)),
           (1201, 601, 8, 1, 2, (2, 4), (0, 0)), (1997, 598, 8, 1, 3, (0, 0), (0, 0)), (4000, 1200, 8, 1, 0, (0, 0), (0, 0))]


@pytest.mark.parametrize("nx,ny,fdorder,physics,L,fwd,adj", CHOICES)
def test_the_librarys_choice(nx, ny, fdorder, physics, L, fwd, adj):
    case = make_case(nx=nx, ny=ny, nt=20, fdorder=fdorder, fw=10, L=L, mode=1, dtinv=5, homogeneous=True, nrec=50, seismo=4)
    g = context(case, False)
    print(f"choice {nx}x{ny} order {fdorder} L {L}", flush=True)
    got, path = forward_and_adjoint(g, case[0])
    assert path == [fwd + (0,), adj + (0,)]
    g.set_tile(64, 4, 1, 1)
    want, path = forward_and_adjoint(g, case[0])
    assert path == [(0, 0, 0)] * 2
    for k, (x, y) in enumerate(zip(got, want)):
        np.testing.assert_array_equal(x, y, err_msg=f"output {k}")


@pytest.mark.parametrize("shape", SHAPES)
def test_engine_rounds_of_every_shape(shape):
    """Forward and adjoint rounds of two shots, one of them in a single row of
    tiles whose height is no multiple of the rows per thread."""
    cases = [make_case(nx=nx, ny=ny, nt=120, fdorder=8, fw=fw, mode=1, dtinv=2, fc=15.0, nrec=nx // 4, seed=nx)
             for nx, ny, fw in [(333, 150, 10), (25, 22, 2)]]
    eng = dnhip.Engine()
    shots = [context(c, False) for c in cases]
    print(f"rounds of shape {shape}", flush=True)
    for phase in (0, 1):
        for g in shots:
            g.set_loop(*shape)
            if phase:
                zero = np.zeros_like(g.seismogram(0))
                g.residuals(zero, zero, None, 1)
            eng.attach(g, phase)
        eng.step(120)
        for g in shots:
            assert eng.status(g) == 0 and g.loop() == shape + (0,)
    for case, g in zip(cases, shots):
        ref = context(case, True)
        ref.forward()
        zero = np.zeros_like(ref.seismogram(0))
        ref.residuals(zero, zero, None, 1)
        ref.adjoint()
        assert np.abs(ref.gradient(0)).max() > 0
        for w in range(3):
            np.testing.assert_array_equal(g.gradient(w), ref.gradient(w), err_msg=f"{case[0].nx} sum {w}")


def test_threads_share_a_kernel():
    """Two contexts in two threads launch one kernel with different amounts of
    LDS, and each launch is accepted."""
    import threading
    ctx = []
    for nx, ny, nt in [(60, 30, 20), (1400, 480, 20)]:
        case = make_case(nx=nx, ny=ny, nt=nt, fdorder=8, fw=10, homogeneous=True)
        g = context(case, False)
        g.set_loop(3, 4)
        g.forward()
        assert g.loop() == (3, 4, 0)
        ctx.append(g)
    paths = [set(), set()]

    def work(k, n):
        for _ in range(n):
            ctx[k].forward()
            paths[k].add(ctx[k].loop())

    print("two threads, one kernel", flush=True)
    ts = [threading.Thread(target=work, args=a) for a in [(0, 300), (1, 100)]]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert paths == [{(3, 4, 0)}] * 2
