"""Set-up work of a shot on the device against its host definition: the model
planes of an elastic P/SV context."""
import numpy as np
import pytest

import dnhip
import orc
from cases import make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("invmat1", [1, 3])
@pytest.mark.parametrize("nx,ny", [(31, 33), (64, 32), (97, 71), (259, 40)])
def test_elastic_model_planes(nx, ny, invmat1, mode):
    """Averages at the edges of the 32 x 32 and 256-cell blocks, with the
    first row and column as the neighbours of the last; cells without shear
    modulus or density; a second model over the first.  The seismograms of
    the run are the oracle's bit for bit."""
    rng = np.random.default_rng(nx)
    case = make_case(nx=nx, ny=ny, nt=60, fw=5, seismo=4, free_surf=0, invmat1=invmat1, mode=mode)
    p, m, src, sig, rec = case
    m = {k: None if v is None else v.copy() for k, v in m.items()}
    for k in ("vp", "vs", "rho"):
        m[k] *= (1.0 + 0.05 * rng.random((nx, ny))).astype(np.float32)
    m["vs"][nx // 2:nx // 2 + 5, 4:9] = 0.0
    m["rho"][-1, -1] = m["rho"][0, -1] = m["rho"][-1, 0] = 0.0
    if invmat1 == 3:
        m["vp"][-1, -1] = m["vp"][0, -1] = m["vp"][-1, 0] = 0.0
        m["vs"][-1, -1] = m["vs"][0, -1] = m["vs"][-1, 0] = 0.0
        m["rho"][-1, -1] = m["rho"][0, -1] = m["rho"][-1, 0] = 2000.0
    dt = np.float32(p.dt * 0.8)
    p = dnhip.Params(**{**p.__dict__, "dt": float(dt)})
    g = dnhip.Context(p)
    g.set_model(np.full((nx, ny), 7.0, np.float32), np.full((nx, ny), 3.0, np.float32),
                np.full((nx, ny), 900.0, np.float32))
    g.set_model(m["vp"], m["vs"], m["rho"])
    g.set_sources(src, sig)
    g.set_receivers(rec)
    print(f"model planes {nx}x{ny} invmat1 {invmat1} mode {mode}", flush=True)
    g.forward()
    o = orc.Oracle(p, m["vp"], m["vs"], m["rho"], prec="f32")
    o.set_sources(src, sig)
    o.set_receivers(rec)
    o.forward()
    for k in range(4):
        assert np.abs(o.seismogram(k)).max() > 0
        np.testing.assert_array_equal(g.seismogram(k), o.seismogram(k))
