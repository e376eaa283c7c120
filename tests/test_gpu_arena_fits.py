"""dn_arena_fits against dn_ctx_create_in: a context whose fit is promised
can be made, with its sources and receivers, in the smallest arena that
promises it (the grid's cell lists are of some hundred kilobytes)."""
import pytest

import dnhip
from cases import make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nrec", [(4000, 1200, 400), (1203, 401, 598), (60, 50, 20)])
def test_promised_context_fits(nx, ny, nrec):
    p, m, src, sig, rec = make_case(nx=nx, ny=ny, nt=12, fdorder=8, fw=10, homogeneous=True, nrec=nrec)
    need = dnhip.estimate_footprint(p, src.shape[1], rec.shape[1])
    for extra in range(0, 8 << 20, 64 << 10):
        arena = dnhip.Arena(need + extra)
        if arena.fits(p, src.shape[1], rec.shape[1]):
            break
        arena.close()
    print(f"arena {nx}x{ny}: {extra >> 10} KB beside the footprint", flush=True)
    g = dnhip.Context(p, arena=arena)
    g.set_model(m["vp"], m["vs"], m["rho"], m["taus"], m["taup"])
    g.set_sources(src, sig)
    g.set_receivers(rec)
    g.close()
    arena.close()
