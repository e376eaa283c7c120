"""A refused dn_set_sources or dn_set_receivers leaves the context without
sources or receivers, not with cell lists of the call before."""
import numpy as np
import pytest

import dnhip
from cases import make_case

pytestmark = pytest.mark.gpu


def context(p, m, arena=None):
    g = dnhip.Context(p, arena=arena)
    g.set_model(m["vp"], m["vs"], m["rho"])
    return g


@pytest.mark.parametrize("sweeps", [False, True])
@pytest.mark.parametrize("stype", [1, 3])
def test_source_outside_the_grid(stype, sweeps):
    p, m, src, sig, rec = make_case(nx=90, ny=60, nt=60, fw=5, seismo=1, stype=stype, nrec=20)
    g = context(p, m)
    if sweeps:
        g.set_tile(64, 4, 1, 1)
    g.set_receivers(rec)
    g.set_sources(src, sig)
    g.forward()
    want = g.seismogram(1)
    assert np.abs(want).max() > 0
    bad = src.copy()
    bad[0] = p.nx + 1
    with pytest.raises(dnhip.DnError) as e:
        g.set_sources(bad, sig)
    assert e.value.code == -1 and "outside" in str(e.value)
    print(f"run after a refused source, sweeps {sweeps}", flush=True)
    g.forward()
    assert np.abs(g.seismogram(1)).max() == 0 and np.abs(g.field(dnhip.F_VX)).max() == 0
    g.set_sources(src, sig)
    g.forward()
    np.testing.assert_array_equal(g.seismogram(1), want)


def test_no_memory_for_points():
    p, m, src, sig, rec = make_case(nx=90, ny=60, nt=200, fw=5, seismo=1, nrec=20)
    arena = dnhip.Arena(dnhip.estimate_footprint(p, 1, 20) + (600 << 10))
    g = context(p, m, arena)
    g.set_receivers(rec)
    g.set_sources(src, sig)
    g.forward()
    want = g.seismogram(1)
    assert np.abs(want).max() > 0
    with pytest.raises(dnhip.DnError) as e:
        g.set_sources(np.repeat(src, 20000, 1), np.repeat(sig, 20000, 0))
    assert e.value.code == -3
    print("run without sources", flush=True)
    g.forward()
    assert np.abs(g.seismogram(1)).max() == 0
    g.set_sources(src, sig)
    many = np.array([[i, j] for i in range(1, 90) for j in range(2, 60)], np.int32).T.copy()
    with pytest.raises(dnhip.DnError) as e:
        g.set_receivers(many)
    assert e.value.code == -3
    print("run without receivers", flush=True)
    g.forward()
    assert np.abs(g.field(dnhip.F_VX)).max() > 0
    g.set_receivers(rec)
    g.forward()
    np.testing.assert_array_equal(g.seismogram(1), want)
    g.close()
    arena.close()
