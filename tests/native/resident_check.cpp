// Host check of the chip-resident loop's geometry (dn_resident_plan.{h,cpp}):
// over many grids, orders and physics, the tiles cover the grid, every access
// stays inside the tile's LDS and the run's mailboxes, every word that is
// waited for is sent by exactly one thread from the cell it stands for, and
// the words are the halo the stencils reach.  Exit status 0 when all hold.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "dn_resident_plan.h"

using namespace dn;

static long fails = 0;
#define CHECK(c)                                                                  \
    do {                                                                          \
        if (!(c) && fails++ < 20) std::fprintf(stderr, "line %d: %s\n", __LINE__, #c); \
    } while (0)

template <int F, int PH, int TW>
static void check(const dn_params &p, const ResPlan &pl)
{
    constexpr int HP = 4 * ((F + 3) / 4), LP = TW + 2 * HP;
    const int nf = res_planes(PH);
    const ResCut cut{pl.gx, pl.gy, pl.tw, pl.th, pl.cap};
    CHECK(pl.tw <= TW && pl.tw % 4 == 0 && pl.tw >= 8 && pl.nthr <= res_maxt(pl.ry, pl.vx, F, p.L) && pl.nthr % 64 == 0 && pl.ncomp <= pl.nthr && pl.tiles() <= 256);
    CHECK((pl.gx - 1) * pl.tw < p.nx && pl.gx * pl.tw >= p.nx && (pl.gy - 1) * pl.th < p.ny && pl.gy * pl.th >= p.ny);
    CHECK(pl.th % pl.ry == 0 && pl.nthx * pl.vx == pl.tw && pl.ncomp == pl.nthx * (pl.th / pl.ry));
    CHECK(pl.cap <= RES_CAP && pl.lds <= 163840);
    // CPML memory: every band cell of a tile has its own place in LDS
    const int np = PH == 2 || PH == 5 ? 2 : 4;
    for (int tile = 0; tile < pl.tiles(); ++tile) {
        const int x0 = tile % pl.gx * pl.tw, y0 = tile / pl.gx * pl.th;
        const int w = std::min(pl.tw, p.nx - x0), h = std::min(pl.th, p.ny - y0);
        const ResBand b = res_band(p.nx, p.ny, p.fw, !p.free_surf, x0, y0, w, h);
        CHECK(b.nx <= pl.ncx && b.ny <= pl.ncy);
        const int FS = LP * (h + 2 * F);
        const size_t fields = (size_t)res_plane_at<F, PH, TW>(nf, FS);
        CHECK(fields < 65536 && fields % 4 == 0);
        const size_t at = (fields + (8 * (2 * p.fw + 1) + 3) / 4 * 4) * 4 + 16;
        CHECK(at % 16 == 0 && at + (size_t)np * ((b.nx ? h * pl.ncx * 4 : 0) + (b.ny ? pl.ncy * pl.tw : 0)) * 4 <= pl.lds);
        for (int tx = 0; tx * 4 < w; ++tx) {
            bool in = false;
            for (int e = 0; e < 4 && tx * 4 + e < w; ++e) {
                const int i = x0 + tx * 4 + e + 1;
                in = in || i <= p.fw || i >= p.nx - p.fw + 1;
            }
            const int id = tx < b.xl ? tx : b.xl + tx - b.xs;
            CHECK(!in || ((tx < b.xl || tx >= b.xs) && id < pl.ncx));
        }
        for (int row = 0; row < h; ++row) {
            const int j = y0 + row + 1;
            const bool up = !p.free_surf && j <= p.fw, in = up || j >= p.ny - p.fw + 1;
            const int id = up ? row : b.yt + row - b.ys;
            CHECK(!in || ((up ? row < b.yt : row >= b.ys) && id >= 0 && id < pl.ncy));
        }
    }
    // the deepest rows and columns a thread's stencil reads
    CHECK(pl.th - pl.ry + F + pl.ry - 1 + F <= pl.th + 2 * F - 1 && TW - 4 + HP + 4 + HP <= LP);
    for (int ex = 0; ex < 2; ++ex) {
        const int nk = ex ? pl.nk_v : pl.nk_s;
        CHECK(nk <= res_ki(F) && nk * pl.nthr >= pl.cap);
        std::vector<long> sent((size_t)pl.tiles() * 2 * pl.cap, -1), want(sent);  // mailbox word -> cell
        long nsent = 0, nwant = 0;
        long expect = 0;
        for (int tile = 0; tile < pl.tiles(); ++tile) {
            const int x0 = tile % pl.gx * pl.tw, y0 = tile / pl.gx * pl.th;
            const int w = std::min(pl.tw, p.nx - x0), h = std::min(pl.th, p.ny - y0);
            CHECK((pl.gx == 1 || w >= F) && h >= F);
            // plane and grid position of an LDS element: the planes whose rows
            // (with halo, but for sxx) hold it
            const int FS = LP * (h + 2 * F);
            std::vector<int> plane_of(res_plane_at<F, PH, TW>(nf, FS), -1);
            for (int f = 0; f < nf; ++f)
                for (int row = res_no_rows(PH, f) ? 0 : -F; row < (res_no_rows(PH, f) ? h : h + F); ++row)
                    for (int col = 0; col < LP; ++col) {
                        int &o = plane_of.at((size_t)(res_plane_at<F, PH, TW>(f, FS) + (row + F) * LP + col));
                        CHECK(o < 0);
                        o = f;
                    }
            for (int o : plane_of) CHECK(o >= 0);
            auto cell = [&](long el) {
                const long plane = plane_of[(size_t)el], in = el - res_plane_at<F, PH, TW>((int)plane, FS);
                const long row = in / LP - F, col = in % LP - HP;
                return (plane * (p.ny + 100) + (y0 + row + 50)) * (p.nx + 100) + (x0 + col + 50);
            };
            auto inside = [&](long el) {
                const long in = el - res_plane_at<F, PH, TW>(plane_of[(size_t)el], FS);
                const long row = in / LP - F, col = in % LP - HP;
                return row >= 0 && row < h && col >= 0 && col < w;
            };
            std::vector<char> got(plane_of.size(), 0);
            for (int t = 0; t < pl.nthr; ++t) {
                Words<F> o;
                res_words<F, PH, TW>(cut, ex, tile, t, pl.nthr, w, h, o);
                for (int k = 0; k < res_ki(F); ++k) {
                    if (k >= nk) CHECK(!(o.rx >> k & 1) && !(o.tx >> k & 1));
                    const long er = o.off[k] & 0xffff, es = o.off[k] >> 16;
                    CHECK(er < (long)got.size() && es < (long)got.size());
                    if (o.rx >> k & 1) {
                        const long word = (long)(tile * 2 + ex) * pl.cap + k * pl.nthr + t;
                        CHECK(!inside(er) && !got[er] && want[word] < 0);
                        got[er] = 1;
                        want[word] = cell(er);
                        ++nwant;
                    }
                    if (o.tx >> k & 1) {
                        CHECK(inside(es) && o.dst[k] < (unsigned long)pl.tiles() * 2 * pl.cap);
                        if (o.dst[k] < sent.size()) {
                            CHECK(sent[o.dst[k]] < 0);
                            sent[o.dst[k]] = cell(es);
                            ++nsent;
                        }
                    }
                }
            }
            const int bx = tile % pl.gx, by = tile / pl.gx;
            const bool has[4] = {bx > 0, bx < pl.gx - 1, by > 0, by < pl.gy - 1};
            for (int side = 0; side < 4; ++side) {
                const Seg s = res_seg<F, PH>(ex, side);
                if (has[side]) expect += (long)(s.na + s.nb) * (side < 2 ? h : w);
                // every halo cell of the segment is among the received ones
                for (int c = 0; has[side] && c < s.na + s.nb; ++c)
                    for (int q = 0; q < (side < 2 ? h : w); ++q) {
                        const int pn = c < s.na ? s.pa : s.pb, cc = c < s.na ? c : c - s.na;
                        const int d = side == 0 || side == 2 ? -1 - cc : (side == 1 ? w : h) + cc;
                        const int row = side < 2 ? q : d, col = side < 2 ? d : q;
                        CHECK(got[(size_t)(res_plane_at<F, PH, TW>(pn, FS) + (row + F) * LP + HP + col)]);
                    }
            }
        }
        CHECK(nwant == expect && nsent == nwant && sent == want);
    }
}

template <int F, int PH>
static bool one(dn_params p)
{
    p.physics = PH;
    p.fdorder = 2 * F;
    const ResPlan pl = res_plan(p, 256, 163840);
    if (!pl.ok) return false;
    if (pl.ry == 1) check<F, PH, res_width(1)>(p, pl);
    if (pl.ry == 2) check<F, PH, res_width(2)>(p, pl);
    if (pl.ry == 3) check<F, PH, res_width(3)>(p, pl);
    return true;
}

// the plans of a launch that holds several grids: a given thread shape in few
// tiles, with the threads of the launch's largest workgroup
template <int F, int PH>
static int packed(dn_params p)
{
    p.physics = PH;
    p.fdorder = 2 * F;
    int n = 0;
    for (int s = 0; s < RES_SHAPES; ++s) {
        const ResPlan least = res_least(p, 163840 - 2048, s);
        if (!least.ok || least.tiles() > 256) continue;
        // no thread shape and budget below it fits
        CHECK(!res_plan(p, least.tiles() - 1, 163840 - 2048, s).ok);
        for (int more : {0, 7}) {
            ResPlan pl = res_plan(p, least.tiles() + more, 163840 - 2048, s);
            CHECK(pl.ok && pl.tiles() <= least.tiles() + more);
            CHECK(pl.ry == res_shapes[s][0] && pl.vx == res_shapes[s][1]);
            if (more) {
                pl.nthr = std::min(pl.nthr + 128, res_maxt(pl.ry, pl.vx, F, p.L));
                pl.nk_s = pl.nk_v = (pl.cap + pl.nthr - 1) / pl.nthr;
            }
            if (pl.ry == 1) check<F, PH, res_width(1)>(p, pl);
            if (pl.ry == 2) check<F, PH, res_width(2)>(p, pl);
            if (pl.ry == 3) check<F, PH, res_width(3)>(p, pl);
            ++n;
        }
    }
    return n;
}

template <int F>
static int orders(const dn_params &p)
{
    return one<F, 1>(p) + one<F, 2>(p) + one<F, 3>(p) + one<F, 5>(p);
}

int main()
{
    const int grids[][2] = {{20, 12}, {32, 8}, {33, 9}, {37, 21}, {64, 64}, {120, 80}, {131, 77}, {400, 200},
                            {500, 174}, {811, 303}, {1237, 431}, {1501, 601}, {1800, 700}, {2000, 600}, {2049, 510},
                            {4000, 1200}, {4000, 80}, {40, 4000}};
    int fit = 0, all = 0;
    for (auto &g : grids) {
        dn_params p{};
        p.nx = g[0];
        p.ny = g[1];
        p.fw = std::min(20, std::min(g[0], g[1]) / 2);
        p.free_surf = g[0] % 2;
        const int n = orders<1>(p) + orders<2>(p) + orders<3>(p) + orders<4>(p) + orders<5>(p) + orders<6>(p);
        std::printf("%d x %d: %d of 24 fit\n", g[0], g[1], n);
        fit += n;
        all += 24;
    }
    std::mt19937 rng(5);
    for (int k = 0; k < 16; ++k) {
        dn_params p{};
        p.nx = 24 + (int)(rng() % 1200);
        p.ny = 10 + (int)(rng() % 700);
        p.fw = std::min(10, std::min(p.nx, p.ny) / 2);
        p.free_surf = k % 2;
        fit += orders<2>(p) + orders<4>(p) + orders<5>(p);
    }
    for (int k = 0; k < 5; ++k) {
        dn_params p{};
        p.nx = 60 + (int)(rng() % 700);
        p.ny = 40 + (int)(rng() % 300);
        p.fw = 10;
        p.free_surf = k % 2;
        fit += packed<2, 1>(p) + packed<4, 1>(p);
    }
    std::printf("%s, %d plans\n", fails ? "resident geometry wrong" : "resident geometry ok", fit);
    return fails ? 1 : 0;
}
