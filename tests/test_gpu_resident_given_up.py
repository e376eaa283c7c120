"""Runs of the chip-resident time loop that are given up leave partial states,
snapshots and sums behind; the repeat by the sweeps has to discard them all.
The workgroup of the first tile leaves after the steps that dn_set_loop gives,
as after a wait that took too long; the others find its flag in their waits.
Every kernel exits normally."""
import numpy as np
import pytest

import dnhip
from cases import make_case
from test_gpu_resident import context, state

pytestmark = pytest.mark.gpu


def gradient_case(L=0, nt=90):
    return make_case(nx=333, ny=150, nt=nt, fdorder=8, fw=10, L=L, mode=1, dtinv=1, homogeneous=True, seismo=4, nrec=60)


def adjoint(g, p):
    rng = np.random.default_rng(3)
    g.set_adjoint_sources(*[(rng.standard_normal((g.ntr, p.nt)) * 1e-6).astype(np.float32) for _ in range(3)])
    g.adjoint()
    return [g.gradient(k) for k in range(3)] + state(g, p)


def same(got, want):
    for k, (x, y) in enumerate(zip(got, want)):
        np.testing.assert_array_equal(x, y, err_msg=f"output {k}")


@pytest.mark.parametrize("shape,L", [((1, 1), 0), ((1, 2), 2), ((2, 4), 0), ((3, 4), 0)])
def test_forward_and_adjoint_repeat(shape, L):
    case = gradient_case(L)
    p = case[0]
    ref = context(case, True)
    ref.forward()
    fwd = state(ref, p)
    adj = adjoint(ref, p)
    assert np.abs(fwd[0]).max() > 0 and np.abs(adj[0]).max() > 0
    print(f"given up: shape {shape} L {L}", flush=True)
    # the forward run given up; the adjoint run reads the repeat's snapshots
    g = context(case, False)
    g.set_loop(*shape, quit=20)
    g.forward()
    assert g.loop() == (0, 0, 1)
    same(state(g, p), fwd)
    g.set_loop(*shape)
    same(adjoint(g, p), adj)
    assert g.loop() == (shape if shape[0] == 1 or L == 0 else (0, 0)) + (1,)
    # the adjoint run given up
    g = context(case, False)
    g.set_loop(*shape)
    g.forward()
    assert g.loop() == shape + (0,)
    g.set_loop(*shape, quit=20)
    same(adjoint(g, p), adj)
    assert g.loop() == (0, 0, 1)
    g.close()


@pytest.mark.parametrize("quit", [20, 2040, 3000, 4200])
def test_run_of_several_launches_repeats(quit):
    """Given up in the first, second and third launch of 2048 steps."""
    case = make_case(nx=200, ny=90, nt=4500, fw=10)
    g, ref = context(case, False), context(case, True)
    g.set_loop(quit=quit)
    print(f"given up: after {quit} of 4500 steps", flush=True)
    g.forward()
    assert g.loop() == (0, 0, 1)
    ref.forward()
    same(state(g, case[0]), state(ref, case[0]))


@pytest.mark.parametrize("beside", [False, True])
@pytest.mark.parametrize("first", [0, 30])
def test_engine_restarts_the_shots_of_its_rounds(first, beside):
    """A round given up in the engine's first or second call; beside it, a
    shot of the sweeps goes on (rounds beside the sweeps are large ones)."""
    sizes = [(333, 150, 90), (1401, 809, 80)] + ([(260, 120, 100)] if beside else [])
    cases = [make_case(nx=nx, ny=ny, nt=nt, fdorder=8, fw=10, seismo=4, homogeneous=True, nrec=nx // 3, seed=k + 1)
             for k, (nx, ny, nt) in enumerate(sizes)]
    shots = [context(c, False) for c in cases]
    if beside:
        shots[2].set_tile(128, 2, 4, 1)
    eng = dnhip.Engine()
    for g in shots:
        eng.attach(g)
    print(f"given up: engine after {first} steps, beside the sweeps {beside}", flush=True)
    if first:
        eng.step(first)
        assert [g.loop()[0] > 0 for g in shots] == [True, True, False][:len(shots)]
    shots[1].set_loop(quit=first + 20)
    eng.step(40)
    assert [g.loop()[1:] for g in shots] == [(0, 1), (0, 1), (0, 0)][:len(shots)]
    eng.run()
    for case, g in zip(cases, shots):
        assert eng.status(g) == 0
        ref = context(case, True)
        ref.forward()
        assert np.abs(ref.field(dnhip.F_VX)).max() > 0
        same(state(g, case[0]), state(ref, case[0]))


def test_runs_after_a_given_up_one():
    """The runs after it take the sweeps at once, two, four and so on, and the
    loop is back when it is set anew."""
    case = make_case(nx=200, ny=90, nt=30, fw=10)
    g = context(case, False)
    g.set_loop(quit=10)
    tries = []
    for _ in range(20):
        g.forward()
        tries.append(g.loop()[2])
    assert tries == [1] * 3 + [2] * 5 + [3] * 9 + [4] * 3
    g.set_loop()
    g.forward()
    assert g.loop() == (1, 1, 4)


def test_shots_attached_after_a_given_up_run():
    case = make_case(nx=200, ny=90, nt=30, fw=10)
    eng = dnhip.Engine()
    g = context(case, False)
    paths = []
    for quit in (10, 0, 0, 0):
        g.set_loop(quit=quit)
        eng.attach(g)
        eng.step(30)
        paths.append(g.loop()[0])
        eng.run()
        assert eng.status(g) == 0
    assert paths == [0, 0, 0, 1] and g.loop()[2] == 1
