"""Work around a shot's time loop on the device against its host definition:
the model planes of an elastic P/SV context, the residuals of its traces."""
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


@pytest.mark.parametrize("nt", [2, 255, 256, 257, 530])
@pytest.mark.parametrize("ntr", [1, 15, 16, 17, 50])
def test_residual_traces(ntr, nt):
    """Edges of the 16-trace, 256-sample pieces: the time integral is one
    float32 chain per trace, so every sample is the host chain's."""
    case = make_case(nx=120, ny=40, nt=nt, fw=5, seismo=1, mode=1, nrec=ntr)
    p, m, src, sig, rec = case
    g = dnhip.Context(p)
    g.set_model(m["vp"], m["vs"], m["rho"])
    g.set_sources(src, sig)
    g.set_receivers(rec)
    g.forward()
    rng = np.random.default_rng(nt + ntr)
    obs = [rng.standard_normal((ntr, nt)).astype(np.float32) for _ in range(2)]
    print(f"residuals of {ntr} traces, {nt} samples", flush=True)
    for w in (1.0, 0.3):
        g.set_residual_weights(w, 1.0)
        l2 = g.residuals(obs[0], obs[1], None, 1)
        want = 0.0
        for k in range(2):
            f = np.float32(w if k == 0 else 1.0)
            s = g.seismogram(k).reshape(ntr, nt) * f
            d = obs[k] * f
            d[:, 0] = s[:, 0]
            x = np.float32(p.dt) * (s - d)
            r = np.zeros_like(x)
            acc = np.zeros(ntr, np.float32)
            for n in range(nt):
                acc = acc + x[:, n]
                r[:, nt - 1 - n] = acc
            np.testing.assert_array_equal(g.adjoint_sources(k).reshape(ntr, nt), r)
            want += float((0.5 * r.astype(np.float64) ** 2).sum())
        # a sum of n positive terms in any order: n roundings at most
        assert abs(l2 - want) <= 2 * ntr * nt * 2.3e-16 * want


@pytest.mark.parametrize("nx,ny,L", [(29, 21, 0), (130, 67, 3)])
def test_state_is_cleared(nx, ny, L):
    """A second run of a context starts from zeros in every field, memory
    variable and CPML array (odd lengths among them)."""
    case = make_case(nx=nx, ny=ny, nt=40, L=L, fw=5, seismo=4, homogeneous=True)
    p, m, src, sig, rec = case
    g = dnhip.Context(p)
    g.set_model(m["vp"], m["vs"], m["rho"], m["taus"], m["taup"])
    g.set_sources(src, sig)
    g.set_receivers(rec)
    print(f"cleared state {nx}x{ny} L {L}", flush=True)
    out = []
    for _ in range(2):
        g.forward()
        out.append([g.field(k) for k in range(7)] + [g.psi(k) for k in range(9)] +
                   [g.memvar(w, l + 1) for w in range(3) for l in range(L)])
    assert np.abs(out[0][0]).max() > 0
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
    g.set_sources(src, 0.0 * sig)
    g.forward()
    assert all(not np.any(g.field(k)) for k in range(7)) and all(not np.any(g.psi(k)) for k in range(9))
    assert all(not np.any(g.memvar(w, l + 1)) for w in range(3) for l in range(L))
