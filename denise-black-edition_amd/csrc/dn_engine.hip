// Multi-shot engine: many independent shots (contexts) advanced together.
//
// Every time step is one velocity launch and one stress launch per group of
// shots that share FD order, relaxation count, direction and tile shapes.
// The kernels read the time step from one device clock plus the offset k of
// the step in the current run of steps (shot step = clock + k - base, base
// fixed when the shot is attached); a run of steps ends with one launch that
// moves the clock on.  So the same launch sequence serves every run: the
// engine can capture a run of steps in a hipGraph once and replay it.  Shots of different grid size and length share the
// launches; a shot that has reached its NT leaves its blocks idle until the
// host detaches it.  Shots can be attached and detached between calls
// (continuous batching); their state stays in their contexts.
//
// Shots whose grids fit are advanced by the chip-resident loop instead, many
// of them in one launch (a round, plan_rounds below): their tiles share the
// CUs, and a launch carries a whole run of steps.  The rounds of a run of
// steps follow each other on the engine's stream, the sweeps after them.
//
// The sweeps' groups, too, need not advance together: each goes through the
// whole run of steps before the next, and a group whose wavefields and
// materials exceed the last-level cache is cut into several that do not.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "dn_ctx.h"
#include "dn_sweep_common.h"

using namespace dn;

namespace {

struct Job {
    dn_ctx *ctx;
    int phase;  // 0 forward, 1 adjoint
    long base;  // engine clock before its first step
    bool sweeps = false;  // its chip-resident run was abandoned, or one before it
    int round = -1;       // the round that carries it, -1: the sweeps
    ResPlan plan;
    ResPoints pts;
    size_t lst = 0;  // position of its point lists (ints)
};

// a launch of the chip-resident loop: shots of one FD order, relaxation
// count, direction and thread shape
struct Round {
    ResPlan shape;  // threads and LDS of the launch
    std::vector<int> jobs;
    int fdoh = 0, sw = 0, tiles = 0;
    size_t words = 0, blk = 0;  // mailbox words, position of its workgroups
};

// Fewest steps of a run that the rounds carry: a launch loads and stores the
// whole state of its shots.  Three 400x200 shots, runs of 8 steps: 13.3 us a
// step (sweeps 25.9), 32 steps 7.2; one 2000x600 shot 22.5 (32.4) and 10.3.
constexpr int RES_MIN_STEPS = 8;
// Shots in the sweeps beside a round: while the sweeps' shots stay within
// the last-level cache (about 4.5e6 cells) a million cells more cost them 10
// us a step, and the round 3.5 + 6 us; past it they need another 14 us.
// 1.1e6 cells beside 1.9e6 in the sweeps: 46.4 us with the round, 47.7
// without, beside 3.7e6 63.6 and 70.8; 0.34e6 beside 1.9e6: 42.5 and 38.8.
// Beside 5.0e6: 1.1e6 90.0 and 100.7, 0.79e6 88.6 and 92.9.
constexpr long RES_LLC_CELLS = 4500000;
constexpr long RES_MIN_CELLS[2] = {1100000, 700000};  // of a round, within the cache and past it
// LDS kept for the point lists of a tile
constexpr size_t RES_PTS_LDS = 2048;

struct Group {
    int fdoh, L, sw;
    Tile tv, ts;
    int off_v = 0, nblk_v = 0, off_s = 0, nblk_s = 0;
    int nfull_v = 0, nfull_s = 0;  // full-tile blocks at the head of each table
    long end = 0;                  // engine clock of its last step
};


}  // namespace

struct dn_engine {
    int device = 0;
    hipStream_t stream = nullptr;
    std::vector<Job> jobs;              // running shots
    std::map<dn_ctx *, int> status;     // last known state per shot
    int *d_clock = nullptr;             // device clock (steps run), abort word of the rounds
    long clock = 0;                     // its value once the queued work is done
    bool inflight = false;              // a launched run not yet waited for
    bool dirty = true;
    std::vector<Group> groups;
    BatchShot *d_shots = nullptr;
    int n_shots = 0, cap_shots = 0;
    BatchBlock *d_blk = nullptr;
    size_t cap_blk = 0;
    int graph_steps = 0;
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    // chip-resident rounds
    ResPool *pool = nullptr;
    std::vector<Round> rounds;
    bool resident = false;  // the sweeps' tables leave the shots of the rounds out
    bool leased = false;    // a launched run holds mailboxes and CUs
    ResRest rest;           // shots attached after a given-up run
    ResLease lease;
    int *d_lst = nullptr;  // point lists
    ResBlock *d_rblk = nullptr;
    ResKernel *d_rtab = nullptr;
    size_t cap_lst = 0, cap_rblk = 0, cap_rtab = 0;

    void drop_graph()
    {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        gexec = nullptr;
        graph = nullptr;
    }
    ~dn_engine()
    {
        (void)hipSetDevice(device);
        if (stream) (void)hipStreamSynchronize(stream);
        drop_graph();
        if (d_clock) (void)hipFree(d_clock);
        if (d_shots) (void)hipFree(d_shots);
        if (d_blk) (void)hipFree(d_blk);
        if (d_lst) (void)hipFree(d_lst);
        if (d_rblk) (void)hipFree(d_rblk);
        if (d_rtab) (void)hipFree(d_rtab);
        if (leased) res_pool_give(pool, lease);
        res_pool_close(pool);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

// a device buffer of at least n elements; the old contents are lost
template <class T>
int grow(T **p, size_t *cap, size_t n)
{
    if (n <= *cap) return DN_OK;
    if (*p) HIP_OK(hipFree(*p));
    *p = nullptr;
    const size_t c = std::max(n, 2 * *cap);
    *cap = 0;
    HIP_OK(hipMalloc((void **)p, sizeof(T) * c));
    *cap = c;
    return DN_OK;
}

// Which shots the chip-resident loop carries, and the rounds it does so in.
// A round takes about 3.5 us a step and 1.5 us per thousand cells of a tile
// (FDORDER 8, elastic: 340 cells 4.0 us, 4690 cells 10.6), so the fewest win:
// shots are packed largest first by the fewest tiles that hold them, and the
// CUs left over are then dealt out in proportion.
int plan_rounds(dn_engine *e)
{
    e->rounds.clear();
    for (Job &j : e->jobs) j.round = -1;
    if (!e->pool) return DN_OK;
    const int ncu = res_pool_cus(e->pool);
    const size_t lds = res_pool_lds(e->pool) - RES_PTS_LDS;
    struct Fit {
        int job, least, need[RES_SHAPES];  // tiles by shape, 0: does not fit
    };
    std::map<std::tuple<int, int, int>, std::vector<Fit>> by;
    long swept = 0;  // cells of the shots left to the sweeps
    for (int k = 0; k < (int)e->jobs.size(); ++k) {
        const Job &j = e->jobs[k];
        Fit f{k, 0, {}};
        if (!j.sweeps && res_applies(j.ctx, j.phase))
            for (int s = 0; s < RES_SHAPES; ++s) {
                if (j.ctx->res_shape >= 0 && s != j.ctx->res_shape) continue;
                const ResPlan pl = res_least(j.ctx->p, lds, s);
                const bool ok = pl.ok && res_compiled(j.ctx->fdoh, j.ctx->a.physics, j.ctx->p.L, j.phase, pl.ry);
                f.need[s] = ok && pl.tiles() <= ncu ? pl.tiles() : 0;
                if (f.need[s] && (!f.least || f.need[s] < f.least)) f.least = f.need[s];
            }
        if (f.least)
            by[std::make_tuple(j.ctx->fdoh, j.ctx->p.L, j.phase)].push_back(f);
        else
            swept += (long)j.ctx->p.nx * j.ctx->p.ny;
    }
    struct Pack {
        std::vector<Fit> fit;
        int shape;
        long cells;
    };
    // the lightest shape in which all shots of a round fit together, or -1
    auto shape_of = [&](const std::vector<Fit> &v) {
        for (int s = 0; s < RES_SHAPES; ++s) {
            int sum = 0;
            bool ok = true;
            for (const Fit &f : v) {
                ok = ok && f.need[s];
                sum += f.need[s];
            }
            if (ok && sum <= ncu) return s;
        }
        return -1;
    };
    std::vector<Pack> packs;
    for (auto &kv : by) {
        auto &v = kv.second;
        std::stable_sort(v.begin(), v.end(), [](const Fit &x, const Fit &y) { return x.least > y.least; });
        const size_t first = packs.size();
        for (const Fit &f : v) {
            size_t k = first;
            for (; k < packs.size(); ++k) {
                std::vector<Fit> with = packs[k].fit;
                with.push_back(f);
                const int s = shape_of(with);
                if (s < 0) continue;
                packs[k].fit.swap(with);
                packs[k].shape = s;
                break;
            }
            if (k == packs.size()) packs.push_back(Pack{{f}, shape_of({f}), 0});
        }
    }
    for (Pack &p : packs)
        for (const Fit &f : p.fit) p.cells += (long)e->jobs[f.job].ctx->p.nx * e->jobs[f.job].ctx->p.ny;
    std::stable_sort(packs.begin(), packs.end(), [](const Pack &x, const Pack &y) { return x.cells < y.cells; });
    for (const Pack &p : packs) {
        if (swept && p.cells < RES_MIN_CELLS[swept + p.cells > RES_LLC_CELLS]) {
            swept += p.cells;
            continue;
        }
        Round r;
        int sum = 0;
        for (const Fit &f : p.fit) sum += f.need[p.shape];
        for (const Fit &f : p.fit) {
            Job &j = e->jobs[f.job];
            const ResPlan pl = res_plan(j.ctx->p, (int)((long)ncu * f.need[p.shape] / sum), lds, p.shape);
            if (!pl.ok) continue;
            res_points(j.ctx, pl, &j.pts);
            if (!res_points_fit(j.ctx, pl, j.pts, j.phase)) continue;
            j.plan = pl;
            j.round = (int)e->rounds.size();
            if (r.jobs.empty()) r.shape = pl;
            r.shape.nthr = std::max(r.shape.nthr, pl.nthr);
            r.shape.lds = std::max(r.shape.lds, res_lds(pl, j.pts, j.phase));
            r.fdoh = j.ctx->fdoh;
            r.sw = j.phase;
            r.tiles += pl.tiles();
            r.words += (size_t)pl.tiles() * 2 * pl.cap;
            r.jobs.push_back(f.job);
        }
        if (!r.jobs.empty()) e->rounds.push_back(r);
    }
    // their point lists and workgroups; neighbouring tiles share an XCD's L2
    std::vector<int> lst;
    std::vector<ResBlock> blk;
    int slot = 0;
    for (Round &r : e->rounds) {
        std::vector<ResBlock> v;
        for (int k : r.jobs) {
            Job &j = e->jobs[k];
            lst.resize((lst.size() + 1) / 2 * 2);
            j.lst = lst.size();
            lst.insert(lst.end(), j.pts.blk.begin(), j.pts.blk.end());
            for (int t = 0; t < j.plan.tiles(); ++t) v.push_back(ResBlock{slot, t});
            ++slot;
        }
        r.blk = blk.size();
        for (int b = 0; b < r.tiles; ++b) blk.push_back(v[(size_t)xcd_tile(b, r.tiles)]);
    }
    if (e->rounds.empty()) return DN_OK;
    int rc;
    if ((rc = grow(&e->d_lst, &e->cap_lst, lst.size())) || (rc = grow(&e->d_rblk, &e->cap_rblk, blk.size()))) return rc;
    HIP_OK(h2d(e->stream, e->d_lst, lst.data(), lst.size() * sizeof(int)));
    HIP_OK(h2d(e->stream, e->d_rblk, blk.data(), blk.size() * sizeof(ResBlock)));
    return DN_OK;
}

// the rounds of `steps` steps from the engine's clock
int launch_rounds(dn_engine *e, int steps)
{
    const int parts = (steps + RES_CHUNK - 1) / RES_CHUNK;
    std::vector<ResKernel> tab;
    unsigned tag = e->lease.tag0;
    for (const Round &r : e->rounds)
        for (int part = 0; part < parts; ++part) {
            res_word *box = e->lease.mbox;
            const int k0 = part * RES_CHUNK, k1 = std::min(k0 + RES_CHUNK, steps);  // of this run
            for (int k : r.jobs) {
                const Job &j = e->jobs[k];
                dn_ctx *c = j.ctx;
                StepCtl ctl = j.phase == 0 ? base_ctl(c, 0, 1) : base_ctl(c, 2, 3);
                ctl.seismo = j.phase == 0 ? c->p.seismo : 0;
                ctl.probe = 1;
                ResPlan pl = j.plan;
                pl.nk_s = pl.nk_v = (pl.cap + r.shape.nthr - 1) / r.shape.nthr;
                ResKernel a{c->a, ctl, c->acq, res_args(c, pl, j.pts, e->d_lst + j.lst, j.phase, c->p.nt), nullptr, nullptr};
                a.r.mbox = box;
                a.r.abort = e->d_clock + 1;
                a.r.tag0 = tag;
                a.r.n0 = (int)(e->clock - j.base) + k0;
                a.r.n1 = std::min((int)(e->clock - j.base) + k1 - 1, c->p.nt);
                box += (size_t)pl.tiles() * 2 * pl.cap;
                tab.push_back(a);
            }
            tag += (unsigned)(k1 - k0 + 2);
        }
    int rc;
    if ((rc = grow(&e->d_rtab, &e->cap_rtab, tab.size()))) return rc;
    HIP_OK(h2d(e->stream, e->d_rtab, tab.data(), tab.size() * sizeof(ResKernel)));
    size_t at = 0;
    int slot = 0;  // of the round's first shot in the workgroups' table
    for (const Round &r : e->rounds) {
        for (int part = 0; part < parts; ++part) {
            ResKernel k = tab[at];
            k.tab = e->d_rtab + at - slot;
            k.blk = e->d_rblk + r.blk;
            if (!res_launch(k, r.shape, r.tiles, r.fdoh, r.sw, res_pool_lds(e->pool), e->stream)) {
                // the rounds already launched run to their end: every shot of
                // the rounds starts over, as after an abandoned wait
                static const int one = 1;
                HIP_OK(h2d(e->stream, e->d_clock + 1, &one, sizeof(int)));
                return DN_OK;
            }
            at += r.jobs.size();
        }
        slot += (int)r.jobs.size();
    }
    return DN_OK;
}

// a shot's state before its first step
int begin_shot(dn_ctx *c, int phase)
{
    int rc;
    if ((rc = zero_state(c))) return rc;
    if (phase == 1) {
        const size_t g = (size_t)c->p.nx * c->p.ny * sizeof(float);
        HIP_OK(hipMemsetAsync(c->wc, 0, g, c->stream));
        HIP_OK(hipMemsetAsync(c->wcu, 0, g, c->stream));
        HIP_OK(hipMemsetAsync(c->wcr, 0, g, c->stream));
    } else {
        c->fwd_complete = false;
        // grad_obj_psv.c:71-76: the energies start at zero for each shot
        if (c->eprecond)
            for (int w = 0; w < 2; ++w)
                HIP_OK(hipMemsetAsync(c->ew[w], 0, (size_t)c->p.nx * c->p.ny * sizeof(float), c->stream));
    }
    HIP_OK(hipStreamSynchronize(c->stream));
    return DN_OK;
}

// Planes that both sweeps of a step read or write, per cell
int state_planes(const dn_ctx *c) { return 10 + (c->p.L ? 3 * c->p.L + 3 : 0); }

// The shots of a group (indices into jobs) that go through a run of steps
// together.  Up to 55e6 plane cells (220 MB) one part is the fastest; more
// are packed into parts of 50e6 (200 MB; the last-level cache has 256 MB).
// Elastic FDORDER 8: 3.7e6 cells 53 us a step, 5.0e6 70, 6.2e6 108, 7.8e6 133
// in one part, where a part within the cache takes 14 us and 10 us per million
// cells; three 4000x1200 grids 270 us a step in one part, 177 in three.
std::vector<std::vector<int>> parts_of(const dn_engine *e, std::vector<int> v)
{
    constexpr long ONE = 55000000, PART = 50000000;
    auto weight = [&](int k) {
        const dn_ctx *c = e->jobs[k].ctx;
        return (long)c->p.nx * c->p.ny * state_planes(c);
    };
    long all = 0;
    for (int k : v) all += weight(k);
    if (all <= ONE) return {v};
    std::stable_sort(v.begin(), v.end(), [&](int a, int b) { return weight(a) > weight(b); });
    std::vector<std::vector<int>> parts;
    std::vector<long> load;
    for (int k : v) {
        size_t s = 0;
        while (s < parts.size() && load[s] + weight(k) > PART) ++s;
        if (s == parts.size()) {
            parts.emplace_back();
            load.push_back(0);
        }
        load[s] += weight(k);
        parts[s].push_back(k);
    }
    return parts;
}

// group the running shots (resident: those no round carries) and upload the
// launch tables of the sweeps
int rebuild(dn_engine *e, bool resident)
{
    HIP_OK(hipStreamSynchronize(e->stream));
    e->drop_graph();
    typedef std::tuple<int, int, int, int, int, int, int, int, int, int, int> Key;
    std::map<Key, std::vector<int>> alike;
    for (int k = 0; k < (int)e->jobs.size(); ++k) {
        if (resident && e->jobs[k].round >= 0) continue;
        const dn_ctx *c = e->jobs[k].ctx;
        const Tile &v = c->tile_v, &s = c->tile_s;
        alike[std::make_tuple(c->fdoh, c->p.L, e->jobs[k].phase, v.tbx, v.by, v.ty, v.vw, s.tbx, s.by, s.ty, s.vw)]
            .push_back(k);
    }
    std::vector<std::vector<int>> by;
    for (const auto &kv : alike)
        for (auto &part : parts_of(e, kv.second)) by.push_back(part);
    std::vector<BatchShot> shots;
    std::vector<BatchBlock> blk;
    e->groups.clear();
    for (const auto &part : by) {
        Group g;
        const dn_ctx *c0 = e->jobs[part[0]].ctx;
        g.fdoh = c0->fdoh;
        g.L = c0->p.L;
        g.sw = e->jobs[part[0]].phase;
        g.tv = c0->tile_v;
        g.ts = c0->tile_s;
        std::vector<BatchBlock> bv, bs, lv, ls;  // full and lean blocks of each sweep
        for (int k : part) {
            const Job &j = e->jobs[k];
            dn_ctx *c = j.ctx;
            g.end = std::max(g.end, j.base + c->p.nt);
            BatchShot b{};
            b.a = c->a;
            const StepCtl base = j.phase == 0 ? base_ctl(c, 0, 1) : base_ctl(c, 2, 3);
            b.cv = base;
            b.cv.seismo = j.phase == 0 ? c->p.seismo : 0;
            b.cv.probe = 1;
            b.cv.mode0_gf2 = j.phase == 0 && c->p.mode > 0 && c->p.grad_form == 2;
            b.cs = b.cv;
            b.cv.ntx = c->tile_v.ntx(c->p.nx);
            b.cv.ntiles = b.cv.ntx * c->tile_v.nty(c->p.ny);
            b.cs.ntx = c->tile_s.ntx(c->p.nx);
            b.cs.ntiles = b.cs.ntx * c->tile_s.nty(c->p.ny);
            b.q = c->acq;
            b.nt_total = c->p.nt;
            b.dtinv = c->p.dtinv;
            b.fwdstore = c->p.mode > 0;
            b.vp1_form = c->p.grad_form == 1 || c->p.grad_form == 2;
            b.sw = j.phase;
            b.ew = j.phase == 0 ? (c->eprecond ? c->ew[0] : nullptr) : (c->eprecond == 1 ? c->ew[1] : nullptr);
            const int idx = (int)shots.size();
            shots.push_back(b);
            const int b0 = (int)j.base;
            const int wv = j.phase == 0 ? 0 : 2, ws = wv + 1;
            for (int t : c->full_h[wv]) bv.push_back(BatchBlock{idx, t, b0, b.nt_total});
            for (int t : c->lean_h[wv]) lv.push_back(BatchBlock{idx, t, b0, b.nt_total});
            for (int t : c->full_h[ws]) bs.push_back(BatchBlock{idx, t, b0, b.nt_total});
            for (int t : c->lean_h[ws]) ls.push_back(BatchBlock{idx, t, b0, b.nt_total});
        }
        g.off_v = (int)blk.size();
        g.nfull_v = (int)bv.size();
        g.nblk_v = (int)(bv.size() + lv.size());
        blk.insert(blk.end(), bv.begin(), bv.end());
        blk.insert(blk.end(), lv.begin(), lv.end());
        g.off_s = (int)blk.size();
        g.nfull_s = (int)bs.size();
        g.nblk_s = (int)(bs.size() + ls.size());
        blk.insert(blk.end(), bs.begin(), bs.end());
        blk.insert(blk.end(), ls.begin(), ls.end());
        e->groups.push_back(g);
    }
    if ((int)shots.size() > e->cap_shots) {
        if (e->d_shots) HIP_OK(hipFree(e->d_shots));
        e->d_shots = nullptr;
        e->cap_shots = std::max<int>((int)shots.size(), 2 * e->cap_shots);
        HIP_OK(hipMalloc((void **)&e->d_shots, sizeof(BatchShot) * e->cap_shots));
    }
    if (blk.size() > e->cap_blk) {
        if (e->d_blk) HIP_OK(hipFree(e->d_blk));
        e->d_blk = nullptr;
        e->cap_blk = std::max(blk.size(), 2 * e->cap_blk);
        HIP_OK(hipMalloc((void **)&e->d_blk, sizeof(BatchBlock) * e->cap_blk));
    }
    if (!shots.empty()) HIP_OK(h2d(e->stream, e->d_shots, shots.data(), sizeof(BatchShot) * shots.size()));
    if (!blk.empty()) HIP_OK(h2d(e->stream, e->d_blk, blk.data(), sizeof(BatchBlock) * blk.size()));
    e->n_shots = (int)shots.size();
    e->resident = resident;
    e->dirty = false;
    return DN_OK;
}

// a run of n steps from the clock's value `from`, then the clock moves on by
// n; a group whose shots end before needs no more launches (from < 0: a run
// that is captured once for any clock)
void enqueue_run(dn_engine *e, int n, long from)
{
    for (const Group &g : e->groups) {
        const int steps = from < 0 ? n : (int)std::min<long>(n, g.end - from + 1);
        for (int k = 0; k < steps; ++k) {
            launch_batch_vel(e->d_shots, e->d_blk + g.off_v, g.nblk_v, g.nfull_v, e->d_clock, k, g.tv, g.fdoh, g.sw, e->stream);
            launch_batch_str(e->d_shots, e->d_blk + g.off_s, g.nblk_s, g.nfull_s, e->d_clock, k, g.ts, g.fdoh, g.L, e->stream);
        }
    }
    launch_batch_clock(e->d_clock, n, e->stream);
}

int capture(dn_engine *e)
{
    HIP_OK(hipStreamBeginCapture(e->stream, hipStreamCaptureModeRelaxed));
    enqueue_run(e, e->graph_steps, -1);
    hipGraph_t g = nullptr;
    HIP_OK(hipStreamEndCapture(e->stream, &g));
    e->graph = g;
    HIP_OK(hipGraphInstantiate(&e->gexec, g, nullptr, nullptr, 0));
    return DN_OK;
}

// shots past their NT leave the engine
int collect(dn_engine *e)
{
    std::vector<Job> still;
    for (const Job &j : e->jobs) {
        if (e->clock - j.base <= j.ctx->p.nt) {
            still.push_back(j);
            continue;
        }
        int nan_step = 0;
        HIP_OK(d2h(e->stream, &nan_step, j.ctx->acq.nan_step, sizeof(int)));
        if (j.phase == 0) j.ctx->fwd_complete = j.ctx->p.mode > 0;
        e->status[j.ctx] = nan_step ? DN_ERR_UNSTABLE : 0;
        e->dirty = true;
    }
    e->jobs.swap(still);
    return DN_OK;
}

}  // namespace

int dn_engine_create(int device, dn_engine **out)
{
    if (!out) return fail(DN_ERR_ARG, "null output pointer");
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev)
        return fail(DN_ERR_ARG, "no such HIP device");
    dn_engine *e = new (std::nothrow) dn_engine();
    if (!e) return fail(DN_ERR_OOM, "host allocation failed");
    e->device = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess) {
        delete e;
        return fail(DN_ERR_HIP, "stream creation failed");
    }
    const int zero[2] = {0, 0};
    if (hipMalloc((void **)&e->d_clock, sizeof zero) != hipSuccess ||
        h2d(e->stream, e->d_clock, zero, sizeof zero) != hipSuccess) {
        delete e;
        return fail(DN_ERR_OOM, "engine clock");
    }
    e->pool = res_pool_open(device);
    *out = e;
    return DN_OK;
}

int dn_engine_destroy(dn_engine *e)
{
    delete e;
    return DN_OK;
}

int dn_engine_set_graph(dn_engine *e, int steps)
{
    if (!e || steps < 0) return fail(DN_ERR_ARG, "bad graph length");
    HIP_OK(hipSetDevice(e->device));
    HIP_OK(hipStreamSynchronize(e->stream));
    e->drop_graph();
    e->graph_steps = steps;
    return DN_OK;
}

int dn_engine_attach(dn_engine *e, dn_ctx *c, int phase)
{
    if (!e || !c || (phase != 0 && phase != 1)) return fail(DN_ERR_ARG, "bad attach request");
    if (c->device != e->device) return fail(DN_ERR_ARG, "context and engine are on different devices");
    if (!c->model_set) return fail(DN_ERR_STATE, "dn_set_model must precede dn_engine_attach");
    if (c->qtype == 5) return fail(DN_ERR_ARG, "moment-tensor shots run through dn_run_forward, not the engine");
    if (c->a.physics != 1) return fail(DN_ERR_ARG, "acoustic, SH and VTI/TTI shots run through dn_run_forward, not the engine");
    for (const Job &j : e->jobs)
        if (j.ctx == c) return fail(DN_ERR_STATE, "context already attached");
    if (phase == 1 && (c->p.mode <= 0 || !c->fwd_complete))
        return fail(DN_ERR_STATE, "adjoint phase needs a finished forward phase with snapshots");
    if (e->clock > (1L << 30)) return fail(DN_ERR_STATE, "engine clock exhausted; create a new engine");
    HIP_OK(hipSetDevice(e->device));
    // tile shapes the multi-shot kernels are compiled for; the caller did not
    // choose them
    int rc;
    const bool chosen = c->sweeps_chosen;
    if (!batch_tile_supported(c->tile_v, 0) && (rc = dn_set_tile(c, 0, 128, 2, 4, 1))) return rc;
    // (elastic groups default to 64,4,2,2: on the 64-shot mix 50.7 Gcell/s
    // against 49.2 with 64,4,1,4 and 42.2 with 64,4,2,1)
    if ((!batch_str_supported(c->tile_s, c->p.L) || (c->p.L == 0 && c->tile_s.ty == 1 && c->tile_s.vw == 1)) &&
        (rc = c->p.L == 0 ? dn_set_tile(c, 1, 64, 4, 2, 2) : dn_set_tile(c, 1, 64, 4, 1, 1)))
        return rc;
    c->sweeps_chosen = chosen;
    if ((rc = begin_shot(c, phase))) return rc;
    Job j;
    j.ctx = c;
    j.phase = phase;
    j.base = e->clock - 1;
    j.sweeps = e->rest.skip();
    e->jobs.push_back(j);
    e->status[c] = 1;
    e->dirty = true;
    return DN_OK;
}

int dn_engine_launch(dn_engine *e, int nsteps)
{
    if (!e || nsteps < 0) return fail(DN_ERR_ARG, "bad step request");
    if (e->inflight) return fail(DN_ERR_STATE, "a launched run is still in flight (dn_engine_wait first)");
    HIP_OK(hipSetDevice(e->device));
    int rc;
    // a shot that the loop no longer takes (its options were changed) leaves its round
    for (const Job &j : e->jobs)
        if (j.round >= 0 && !res_applies(j.ctx, j.phase)) e->dirty = true;
    if (e->jobs.empty() || nsteps == 0) return DN_OK;
    if (e->dirty && (rc = plan_rounds(e))) return rc;
    // no more steps than the longest remaining shot needs
    long need = 0;
    for (const Job &j : e->jobs) need = std::max<long>(need, j.ctx->p.nt - (e->clock - j.base) + 1);
    int left = (int)std::min<long>(nsteps, need);
    bool resident = !e->rounds.empty() && left >= RES_MIN_STEPS;
    if (resident) {
        int tiles = 0;
        size_t words = 0;
        for (const Round &r : e->rounds) {
            tiles = std::max(tiles, r.tiles);
            words = std::max(words, r.words);
        }
        // (every launch draws its own tags)
        const unsigned long tags = (unsigned long)res_tags(left) * e->rounds.size();
        e->leased = tags < 0x7fffffffUL && res_pool_take(e->pool, tiles, words, (unsigned)tags, &e->lease);
        resident = e->leased;
    }
    const bool changed = e->dirty || resident != e->resident;
    e->inflight = true;
    if (changed && (rc = rebuild(e, resident))) return rc;
    for (const Job &j : e->jobs) {
        const bool in = resident && j.round >= 0;
        j.ctx->ran_ry = in ? j.plan.ry : 0;
        j.ctx->ran_vx = in ? j.plan.vx : 0;
    }
    if (resident && (rc = launch_rounds(e, left))) return rc;
    e->clock += left;
    // a graph is captured only for a set of shots that has already run
    // unchanged once: capture and instantiation cost milliseconds of host
    // time, which a set that changes at every call (a request stream) would
    // pay each time while plain launches overlap the GPU work
    if (e->graph_steps > 0 && left >= e->graph_steps && (e->gexec || !changed) && !e->groups.empty()) {
        if (!e->gexec && (rc = capture(e))) return rc;
        for (; left >= e->graph_steps; left -= e->graph_steps) HIP_OK(hipGraphLaunch(e->gexec, e->stream));
    }
    if (left > 0) enqueue_run(e, left, e->clock - left);
    HIP_OK(hipGetLastError());
    return DN_OK;
}

int dn_engine_wait(dn_engine *e, int *running)
{
    if (!e) return fail(DN_ERR_ARG, "null engine");
    if (e->inflight) {
        HIP_OK(hipSetDevice(e->device));
        e->inflight = false;
        HIP_OK(hipStreamSynchronize(e->stream));
        int rc;
        if (e->leased) {
            res_pool_give(e->pool, e->lease);
            e->leased = false;
            int word[2] = {0, 0};
            HIP_OK(d2h(e->stream, word, e->d_clock, sizeof word));
            if (!word[1]) {
                e->rest.finished();
            } else {
                e->rest.given_up();
                // the workgroups gave up waiting for each other: the shots of
                // the rounds start over, in the sweeps
                word[1] = 0;
                HIP_OK(h2d(e->stream, e->d_clock + 1, word + 1, sizeof(int)));
                for (Job &j : e->jobs) {
                    if (j.round < 0) continue;
                    j.ctx->ran_ry = j.ctx->ran_vx = 0;
                    ++j.ctx->given_up;
                    if ((rc = begin_shot(j.ctx, j.phase))) return rc;
                    j.sweeps = true;
                    j.base = e->clock - 1;
                }
                e->dirty = true;
            }
        }
        if ((rc = collect(e))) return rc;
    }
    if (running) *running = (int)e->jobs.size();
    return DN_OK;
}

int dn_engine_step(dn_engine *e, int nsteps, int *running)
{
    const int rc = dn_engine_launch(e, nsteps);
    return rc ? rc : dn_engine_wait(e, running);
}

int dn_engine_status(dn_engine *e, dn_ctx *c, int *status)
{
    if (!e || !c || !status) return fail(DN_ERR_ARG, "bad status request");
    auto it = e->status.find(c);
    if (it == e->status.end()) return fail(DN_ERR_ARG, "context was never attached to this engine");
    *status = it->second;
    return DN_OK;
}

int dn_engine_forget(dn_engine *e, dn_ctx *c)
{
    if (!e || !c) return fail(DN_ERR_ARG, "bad request");
    for (const Job &j : e->jobs)
        if (j.ctx == c) return fail(DN_ERR_STATE, "context still running");
    e->status.erase(c);
    return DN_OK;
}
