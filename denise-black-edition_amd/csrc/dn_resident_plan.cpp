// The cut of a grid for the chip-resident time loop.
#include "dn_resident_plan.h"

#include <algorithm>

namespace dn {

static ResBand band(const dn_params &p, const ResPlan &q, int bx, int by)
{
    const int x0 = bx * q.tw, y0 = by * q.th;
    return res_band(p.nx, p.ny, p.fw, !p.free_surf, x0, y0, std::min(q.tw, p.nx - x0), std::min(q.th, p.ny - y0));
}

namespace {
// rows of tiles that p's grid can be cut into with the threads of a shape:
// each fitting cut goes to take(plan, cost) until that returns false
struct Cut {
    const dn_params &p;
    size_t lds_max;
    int F, HP, n, nf, ry, maxt;
    ResPlan q;

    Cut(const dn_params &pp, size_t lds, int shape) : p(pp), lds_max(lds)
    {
        F = p.fdorder / 2;
        HP = 4 * ((F + 3) / 4);
        const int phys = p.physics == 0 ? 1 : p.physics;
        n = phys == 2 || phys == 5 ? 1 : 2;  // differenced planes per tile edge
        nf = res_planes(phys);
        ry = res_shapes[shape][0];
        maxt = res_maxt(ry, res_shapes[shape][1], F, p.L);
        q.ry = ry;
        q.vx = res_shapes[shape][1];
        // the widest tile whose last column is no narrower than the stencil's
        // reach: the halo of a tile comes from its direct neighbour alone
        for (q.tw = res_width(ry); q.tw >= 8; q.tw -= 4) {
            q.gx = (p.nx + q.tw - 1) / q.tw;
            if (q.gx == 1 || p.nx - (q.gx - 1) * q.tw >= F) break;
        }
        // (a cell in both bands of an axis has two memory variables per derivative there)
        if (ry > res_rows(F, phys, p.L, 0) || p.ny < F || p.nx < 2 * p.fw || p.ny < 2 * p.fw) q.tw = 0;
        q.nthx = q.tw / q.vx;
    }
    bool any() const { return q.tw >= 8; }
    // the tile height of gy balanced rows
    int height(int gy) const { return ((p.ny + gy - 1) / gy + ry - 1) / ry * ry; }
    bool too_tall(int th) const { return q.nthx * (th / ry) > maxt; }

    // gy rows of tiles: tiles of one height, the last row shorter where the
    // balanced height does not fit: its corner tiles hold the CPML memory of
    // both axes
    bool rows(int gy)
    {
        for (q.th = height(gy); !too_tall(q.th) && (gy - 1) * q.th < p.ny; q.th += ry) {
            q.gy = (p.ny + q.th - 1) / q.th;
            if (q.th < F || p.ny - (q.gy - 1) * q.th < F) continue;
            q.ncomp = q.nthx * (q.th / ry);
            q.cap = n * (2 * F - 1) * (q.tw + q.th);
            // a thread more for the exchange costs nothing while the CU has idle SIMDs
            q.nthr = std::max((q.ncomp + 63) / 64 * 64, 256);
            while (q.nthr < maxt && q.nthr * res_ki(F) < q.cap) q.nthr += 64;
            if (q.nthr * res_ki(F) < q.cap || q.cap > RES_CAP) continue;
            q.nk_s = q.nk_v = (q.cap + q.nthr - 1) / q.nthr;
            q.ncx = q.ncy = 0;
            for (int k = 0; k < q.gx; ++k) q.ncx = std::max(q.ncx, band(p, q, k, 0).nx);
            for (int k = 0; k < q.gy; ++k) q.ncy = std::max(q.ncy, band(p, q, 0, k).ny);
            q.lds = 0;
            for (int by = 0; by < q.gy; ++by)
                for (int bx = 0; bx < q.gx; ++bx) {
                    const ResBand b = band(p, q, bx, by);
                    const int h = std::min(q.th, p.ny - by * q.th), LP = res_width(ry) + 2 * HP;
                    const int rows = nf * (h + 2 * F) - (nf == 5 ? 2 * F : 0);
                    const size_t prof = (size_t)(8 * (2 * p.fw + 1) + 3) / 4 * 4;
                    const size_t psi_x = b.nx ? (size_t)2 * n * h * q.ncx * 4 : 0, psi_y = b.ny ? (size_t)2 * n * q.ncy * q.tw : 0;
                    // threads whose last rows lie below the tile read them too, and
                    // drop what they get: rows past the last plane, rows past the x memory
                    const size_t below = (size_t)((h + ry - 1) / ry * ry - h), fields = (size_t)rows * LP;
                    const size_t behind = prof + std::max(psi_x + psi_y, psi_x + (b.nx ? below * q.ncx * 4 : 0));
                    q.lds = std::max(q.lds, (fields + std::max(behind, below * LP)) * sizeof(float) + 16);
                }
            if (q.lds > lds_max) continue;
            q.ok = true;
            return true;
        }
        q.ok = false;
        return false;
    }
};
}  // namespace

ResPlan res_plan(const dn_params &p, int ncu, size_t lds_max, int shape)
{
    ResPlan best;
    // The fewest cells per thread that fit: more waves share a CU's four SIMDs
    // and hide each other's latencies.  FDORDER 8 elastic steps: 500x174 4.0 us
    // with 1 x 1 cells per thread, 4.8 with 1 x 2, 6.3 with 1 x 4, 7.4 with
    // 2 x 4, 9.3 with 3 x 4; 1000x400 6.3 with 1 x 2, 7.8 with 1 x 4, 7.7 with
    // 2 x 4, 9.5 with 3 x 4; 1500x600 8.6 with 2 x 4, 10.3 with 3 x 4.
    for (int s = shape < 0 ? 0 : shape; s < (shape < 0 ? RES_SHAPES : shape + 1) && !best.ok; ++s) {
        Cut c(p, lds_max, s);
        double cost = 0.0;
        if (!c.any()) continue;
        for (int gy = std::min(ncu / c.q.gx, p.ny); gy >= 1 && !c.too_tall(c.height(gy)); --gy) {
            if (!c.rows(gy)) continue;
            // waves per SIMD, then the halo words
            const double k = ((c.q.ncomp + 63) / 64 + 3) / 4 + 0.0005 * c.q.cap;
            if (!best.ok || k < cost) {
                best = c.q;
                cost = k;
            }
        }
    }
    return best;
}

ResPlan res_least(const dn_params &p, size_t lds_max, int shape)
{
    Cut c(p, lds_max, shape);
    if (!c.any()) return ResPlan();
    const int most = std::max(c.maxt / c.q.nthx * c.ry, 1);  // rows of a tile
    for (int gy = std::max((p.ny + most - 1) / most, 1); gy <= p.ny; ++gy) {
        if (c.height(gy) < c.F) break;
        if (c.rows(gy)) return c.q;
    }
    return ResPlan();
}

}  // namespace dn
