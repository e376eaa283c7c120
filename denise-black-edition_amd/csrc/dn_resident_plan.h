// Chip-resident time loop (dn_resident.inc): the cut of a grid into one tile
// per CU, and which halo words every thread of a tile sends and receives.
// Plain C++ shared by the host, the kernels and the CPU check of the plan.
#pragma once
#include "dn_internal.h"

#ifdef __HIP__
#define DN_HD __host__ __device__ __forceinline__
#define DN_UNROLL _Pragma("unroll")
#else
#define DN_HD inline
#define DN_UNROLL
#endif

namespace dn {

// A thread owns RY rows of VX columns: 1 x 1, 1 x 2 or 1 x 4 in tiles up to
// 32 columns wide, 2 x 4 or 3 x 4 in tiles up to 64 or 72 wide; the
// widest tile fixes the LDS pitch at compile time.  A workgroup has at most as
// many threads as leave each the registers its shape asks for.  1 x 2 at
// orders up to 8 has more: 128 registers a thread, and it spills up to 133
// (elastic, order 8, 23 forward and 97 adjoint).  More waves still win over
// more columns: 1000x400, order 8, forward and adjoint steps 6.7 and 7.9 us with
// 1 x 2, 8.2 and 9.8 with 1 x 4; one mechanism 7.7, 8.9 and 8.6, 9.8; two 8.3, 10.0
// and 9.2, 10.1; with three they do not (9.7, 11.5 and 9.6, 10.4).
constexpr int res_maxt(int ry, int vx, int F, int L)
{
    return ry > 1 ? 512 : vx == 1 ? 1024 : vx == 2 ? (F <= 4 ? 1024 : 768) : (F <= 4 && L == 0 ? 768 : 512);
}
// Rows per thread, at most (ph: physics, sw: 0 forward, 1 adjoint).  Three
// relaxation mechanisms (nine memory variables per cell) spill with several
// rows: the sweeps were as fast or faster.  So do viscoelastic adjoint runs
// (168 to 345 registers), and a trial build of one with three mechanisms and
// two rows ended in a memory fault.  Its source keeps within bounds when it is
// run on the host (tests/native/resident_exec.cpp), so the cause lies in what
// was compiled and is not known: kernels with several rows that spill 100
// registers or more are left out, but for the two of order 8 that have long
// been run and tested (two mechanisms forward 147, TTI adjoint 126).  Left out:
// three rows in elastic and VTI adjoint runs (103 to 153 registers) and in TTI
// forward runs (202, 217) of orders 10 and 12, two and three in TTI adjoint
// runs of those (155 to 271), three in TTI adjoint runs of orders 2 to 6 (73,
// 113, 110), three in forward runs with two mechanisms of all orders but 8
// (145 to 228).
// Two mechanisms, forward, order 8: 2000x600 27 us a step against 31 in the
// sweeps, 1500x400 16 against 20.
constexpr int res_rows(int F, int ph, int L, int sw)
{
    if (L > 0) return L > 2 || sw ? 1 : L == 2 && F != 4 ? 2 : 3;
    if (ph == 4) return sw && F != 4 ? (F > 4 ? 1 : 2) : F > 4 ? 2 : 3;
    return (ph == 1 || ph == 3) && F > 4 ? 3 - sw : 3;
}
constexpr int res_width(int ry) { return ry == 1 ? 32 : ry == 2 ? 64 : 72; }
constexpr int RES_ENT = 256;     // sources and receivers of one tile and sweep kept in LDS, at most
constexpr int res_ki(int F) { return F <= 4 ? 4 : 6; }  // halo words per thread and exchange, at most
constexpr int RES_CAP = 3072;                           // ... per tile and exchange
// polls before a wait is given up: at the first exchange of a launch (its
// workgroups may still wait for CUs that other work holds: about 20 ms) and
// later (about a second; workgroups that answered once stay resident)
constexpr int RES_SPIN_FIRST = 1 << 14;
constexpr int RES_SPIN = 1 << 20;
constexpr int RES_CHUNK = 2048;  // time steps per launch

// A run that was given up cost its waits, 20 ms and more, and the next one
// would too while other work (another process's loop) holds the CUs: after
// the k-th in a row, 2^k runs, 64 at most, take the sweeps before another try.
struct ResRest {
    int row = 0, left = 0;
    // is this run one of those
    bool skip()
    {
        if (left == 0) return false;
        --left;
        return true;
    }
    void given_up()
    {
        if (row < 6) ++row;
        left = 1 << row;
    }
    void finished() { row = 0; }
};

// the cut of a grid: gx x gy tiles of tw x th cells (tw a multiple of 4; the
// last ones of a row or column may be smaller), nthx x (th / ry) threads owning vx x ry
// cells each, nthr threads in all
struct ResPlan {
    bool ok = false;
    int ry = 1, vx = 4, tw = 0, th = 0, gx = 0, gy = 0, nthx = 0, ncomp = 0, nthr = 0;
    int nk_s = 0, nk_v = 0, cap = 0;  // words per thread, words per tile and exchange
    int ncx = 0, ncy = 0;  // 4-column groups / rows with CPML cells, at most, in a tile
    size_t lds = 0;  // without the point lists
    int tiles() const { return gx * gy; }
};

// LDS planes of a physics
inline int res_planes(int physics) { return physics == 2 || physics == 5 ? 3 : 5; }

// the plan of a grid on a device with ncu CUs and lds_max bytes of LDS per
// workgroup (ok = false: the grid does not fit, in tiles as wide as the shape
// allows); shape: one entry of
// res_shapes, or -1 for the lightest that fits
ResPlan res_plan(const dn_params &p, int ncu, size_t lds_max, int shape = -1);
// the plan of that shape with the fewest tiles
ResPlan res_least(const dn_params &p, size_t lds_max, int shape);
// rows and columns per thread, from the lightest
constexpr int RES_SHAPES = 5;
constexpr int res_shapes[RES_SHAPES][2] = {{1, 1}, {1, 2}, {1, 4}, {2, 4}, {3, 4}};
// LDS planes: vx, vy and the stresses (acoustic: vx, vy, p; SH: vz, sxz, syz)
enum { PL_VX = 0, PL_VY = 1, PL_SXX = 2, PL_SYY = 3, PL_SXY = 4 };
enum { PL_P = 2 };
enum { PL_VZ = 0, PL_SXZ = 1, PL_SYZ = 2 };

// sxx is differenced along x alone: its plane has no halo rows
DN_HD constexpr bool res_no_rows(int ph, int plane) { return ph != 2 && ph != 5 && plane == PL_SXX; }
// LDS element of a plane whose rows start F rows before the tile; FS: floats
// of a plane with halo rows.  The number of planes gives the end of them.
template <int F, int PH, int TW>
DN_HD constexpr int res_plane_at(int plane, int FS)
{
    const int gap = F * (TW + 8 * ((F + 3) / 4));
    if (PH == 2 || PH == 5) return plane * FS;
    // vx, vy, syy, sxy in full, sxx last
    return plane == PL_SXX ? 4 * FS - gap : plane == 5 ? 5 * FS - 2 * gap : (plane > PL_SXX ? plane - 1 : plane) * FS;
}

// the planes and halo widths that the velocity update (ex 0) or the stress
// update (ex 1) reads across a tile edge; side 0 left, 1 right, 2 up, 3 down
struct Seg {
    int pa, na, pb, nb;
};
template <int F, int PH>
DN_HD constexpr Seg res_seg(int ex, int side)
{
    const bool lo = side == 0 || side == 2, x = side < 2;
    // backward differences reach F cells to the low side and F-1 to the high
    // side, forward ones the other way round
    const int bw = lo ? F : F - 1, fwd = lo ? F - 1 : F;
    if (PH == 2) {
        if (ex == 0) return Seg{PL_P, fwd, 0, 0};
        return x ? Seg{PL_VX, bw, 0, 0} : Seg{PL_VY, bw, 0, 0};
    }
    if (PH == 5) {
        if (ex == 0) return x ? Seg{PL_SXZ, bw, 0, 0} : Seg{PL_SYZ, bw, 0, 0};
        return Seg{PL_VZ, fwd, 0, 0};
    }
    if (ex == 0) return x ? Seg{PL_SXX, fwd, PL_SXY, bw} : Seg{PL_SYY, fwd, PL_SXY, bw};
    return x ? Seg{PL_VX, bw, PL_VY, fwd} : Seg{PL_VX, fwd, PL_VY, bw};
}

// CPML cells of a tile (w x h cells after x0, y0): its 4-column groups
// 0..xl-1 and xs.. reach into the x bands, its rows 0..yt-1 and ys.. into
// the y bands
struct ResBand {
    int xl, xs, nx, yt, ys, ny;  // nx, ny: groups and rows with band cells
};
DN_HD ResBand res_band(int NX, int NY, int fw, bool top, int x0, int y0, int w, int h)
{
    ResBand b;
    const int groups = (w + 3) / 4;
    const int l = fw - x0 < w ? fw - x0 : w;
    b.xl = l > 0 ? (l + 3) / 4 : 0;
    const int r = NX - fw - x0;  // columns before the right band
    b.xs = r >= w ? groups : r > 0 ? r / 4 : 0;
    if (b.xs < b.xl) b.xs = b.xl;
    b.nx = b.xl + groups - b.xs;
    const int u = top ? (fw - y0 < h ? fw - y0 : h) : 0;
    b.yt = u > 0 ? u : 0;
    const int d = NY - fw - y0;
    b.ys = d >= h ? h : d > 0 ? d : 0;
    if (b.ys < b.yt) b.ys = b.yt;
    b.ny = b.yt + h - b.ys;
    return b;
}

// the cut as the kernels know it
struct ResCut {
    int gx, gy, tw, th, cap;
};

// the halo words of one exchange that a thread carries
template <int F>
struct Words {
    unsigned off[res_ki(F)];  // LDS element: low half where it is received, high half where it is sent from
    unsigned dst[res_ki(F)];  // mailbox word of the neighbour it is sent to
    unsigned rx, tx;       // bit k: word k is received / sent
};

template <int F, int PH, int TW>
DN_HD void res_words(const ResCut &cut, int ex, int tile, int t, int nthr, int w, int h, Words<F> &o)
{
    constexpr int HP = 4 * ((F + 3) / 4), LP = TW + 2 * HP;
    const int gx = cut.gx, gy = cut.gy, tw = cut.tw, th = cut.th, cap = cut.cap;
    const int FS = LP * (h + 2 * F);
    const int bx = tile % gx, by = tile / gx;
    const bool has[4] = {bx > 0, bx < gx - 1, by > 0, by < gy - 1};
    const int nbr[4] = {tile - 1, tile + 1, tile - gx, tile + gx};
    o.rx = o.tx = 0;
DN_UNROLL
    for (int k = 0; k < res_ki(F); ++k) {
        o.off[k] = 0;
        o.dst[k] = 0;
        const int q = k * nthr + t;
        int rest = q;
        bool done = false;
DN_UNROLL
        for (int side = 0; side < 4; ++side) {
            const Seg s = res_seg<F, PH>(ex, side);
            const int n = s.na + s.nb, len = side < 2 ? th : tw;
            if (!done && rest < n * len) {
                done = true;
                // along a column edge the words of one row are adjacent,
                // along a row edge the columns are
                const int c = side < 2 ? rest % n : rest / len;
                const int p = side < 2 ? rest / n : rest % len;
                const int plane = res_plane_at<F, PH, TW>(c < s.na ? s.pa : s.pb, FS);
                const int cc = c < s.na ? c : c - s.na, nn = c < s.na ? s.na : s.nb;
                const bool in = p < (side < 2 ? h : w);
                // receiver's and sender's position across the edge
                int rr, rs;
                if (side == 0 || side == 2) {
                    rr = cc - nn;
                    rs = (side == 0 ? w : h) + cc - nn;
                } else {
                    rr = (side == 1 ? w : h) + cc;
                    rs = cc;
                }
                const int row_r = side < 2 ? p : rr, col_r = side < 2 ? rr : p;
                const int row_s = side < 2 ? p : rs, col_s = side < 2 ? rs : p;
                const unsigned fr = (unsigned)(plane + (row_r + F) * LP + HP + col_r);
                const unsigned fs = (unsigned)(plane + (row_s + F) * LP + HP + col_s);
                const int opp = side ^ 1;
                const bool rx = in && has[side], tx = in && has[opp];
                o.off[k] = (rx ? fr : 0u) | ((tx ? fs : 0u) << 16);
                if (rx) o.rx |= 1u << k;
                if (tx) {
                    o.tx |= 1u << k;
                    o.dst[k] = (unsigned)(nbr[opp] * 2 + ex) * (unsigned)cap + (unsigned)q;
                }
            }
            if (!done) rest -= n * len;
        }
    }
}


}  // namespace dn
