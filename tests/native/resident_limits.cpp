// Host check of the chip-resident loop's plans with relaxation mechanisms:
// threads within what their kernels are compiled for, and LDS up to the last
// element that a thread of any tile reads, rows below the tile included.
// Exit status 0 when all hold.
#include <algorithm>
#include <cstdio>
#include <random>

#include "dn_resident_plan.h"

using namespace dn;

static long fails = 0, plans = 0;
#define CHECK(c)                                                                  \
    do {                                                                          \
        if (!(c) && fails++ < 20) std::fprintf(stderr, "line %d: %s\n", __LINE__, #c); \
    } while (0)

// the last float (and one) that the threads of a tile read
template <int F, int PH, int TW>
static size_t last(const dn_params &p, const ResPlan &pl, int tile)
{
    constexpr int HP = 4 * ((F + 3) / 4), LP = TW + 2 * HP, K = 4 * ((F + 3) / 4);
    const int x0 = tile % pl.gx * pl.tw, y0 = tile / pl.gx * pl.th;
    const int w = std::min(pl.tw, p.nx - x0), h = std::min(pl.th, p.ny - y0), FS = LP * (h + 2 * F);
    const int nf = res_planes(PH), np = nf == 3 ? 2 : 4;
    const int row = (h - 1) / pl.ry * pl.ry + pl.ry - 1;          // of the last thread
    const int col = (w - 1) / pl.vx * pl.vx + pl.vx - 1;
    size_t end = 0;
    for (int f = 0; f < nf; ++f) {
        const int y = res_no_rows(PH, f) ? 0 : F;
        end = std::max(end, (size_t)res_plane_at<F, PH, TW>(f, FS) + (row + F + y) * LP + HP + col + 1);
        end = std::max(end, (size_t)res_plane_at<F, PH, TW>(f, FS) + (row + F) * LP + HP + col + K + 1);
    }
    const size_t psi = (size_t)res_plane_at<F, PH, TW>(nf, FS) + (8 * (2 * p.fw + 1) + 3) / 4 * 4 + 4;
    const ResBand b = res_band(p.nx, p.ny, p.fw, !p.free_surf, x0, y0, w, h);
    const size_t xf = b.nx ? (size_t)h * pl.ncx * 4 : 0;
    if (b.nx) end = std::max(end, psi + (np - 1) * xf + (size_t)row * pl.ncx * 4 + pl.ncx * 4);
    if (b.ny) end = std::max(end, psi + np * xf + (size_t)np * pl.ncy * pl.tw);
    return end;
}

template <int F, int PH>
static void one(dn_params p, int budget, int shape)
{
    p.physics = PH;
    p.fdorder = 2 * F;
    for (const ResPlan &pl : {res_plan(p, budget, 163840, shape), shape < 0 ? ResPlan() : res_least(p, 161792, shape)}) {
        if (!pl.ok) continue;
        ++plans;
        CHECK(pl.ry <= res_rows(F, PH, p.L, 0));
        CHECK(pl.nthr % 64 == 0 && pl.nthr <= res_maxt(pl.ry, pl.vx, F, p.L));
        CHECK(pl.ncomp <= pl.nthr && pl.nk_s <= res_ki(F) && pl.nk_v <= res_ki(F));
        for (int t = 0; t < pl.tiles(); ++t) {
            const size_t end = pl.ry == 1   ? last<F, PH, res_width(1)>(p, pl, t)
                               : pl.ry == 2 ? last<F, PH, res_width(2)>(p, pl, t)
                                            : last<F, PH, res_width(3)>(p, pl, t);
            CHECK(end * sizeof(float) <= pl.lds && pl.lds <= 163840);
        }
    }
}

int main()
{
    std::mt19937 rng(11);
    for (int k = 0; k < 400; ++k) {
        dn_params p{};
        const bool large = k % 4 == 0;
        p.nx = 13 + (int)(rng() % (large ? 2000 : 200));
        p.ny = 13 + (int)(rng() % (large ? 600 : 90));
        p.fw = std::min((int)(rng() % 21), std::min(p.nx, p.ny) / 2);
        p.free_surf = k % 2;
        for (int L = 0; L < 4; ++L) {
            p.L = L;
            const int budget = large ? 256 : 1 + (int)(rng() % 60), shape = (int)(rng() % 6) - 1;
            one<1, 1>(p, budget, shape);
            one<2, 1>(p, budget, shape);
            one<3, 1>(p, budget, shape);
            one<4, 1>(p, budget, shape);
            one<5, 1>(p, budget, shape);
            one<6, 1>(p, budget, shape);
        }
        p.L = 0;
        one<4, 2>(p, 256, k % 6 - 1);
        one<5, 4>(p, 256, k % 6 - 1);
        one<2, 5>(p, 256, k % 6 - 1);
    }
    std::printf("%s, %ld plans\n", fails ? "resident limits wrong" : "resident limits ok", plans);
    return fails || plans < 1000 ? 1 : 0;
}
