// Host execution of the chip-resident loop's kernel (dn_resident.inc, rewritten
// for g++ by test_resident_exec_host.py): every thread of every workgroup is a
// fiber, LDS is a heap block of exactly the launch's size and every plane one
// of its own size, so the address sanitizer sees each access that leaves them
// and the alignment check each vector that is not aligned.  For one stencil
// half-order (CF), physics (CPH), number of mechanisms (CL) and direction
// (CSW) all thread shapes advance the same states, in plans of several tile
// counts, and have to give the same bits; so has a run cut into two launches.
// Exit status 0 when all hold.
#include <sanitizer/asan_interface.h>
#include <sanitizer/common_interface_defs.h>
#include <sys/mman.h>
#include <ucontext.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <map>
#include <memory>
#include <random>
#include <vector>

// ---------------------------------------------------------------- the device, as far as the kernel knows it
#define __device__
#define __host__
#define __global__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define address_space(n)
#define ext_vector_type(n) vector_size((n) * 4)
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, o, s) (*(p))
#define __hip_atomic_store(p, v, o, s) (*(p) = (v))
#define __builtin_nontemporal_load(p) (*(p))
#define __builtin_nontemporal_store(v, p) (*(p) = (v))
#define __builtin_isfpclass(x, m) ((x) == 0.0f || std::isinf(x))
#define __builtin_amdgcn_s_waitcnt(n) ((void)0)
#define __builtin_amdgcn_sched_barrier(n) ((void)0)
#define __builtin_amdgcn_kernarg_segment_ptr() ((const void *)host_kernel)
#define __ballot(c) ((void)(c), 1ull)  // a wavefront's bit is set if any thread's is: the threads test their own
#define __syncthreads() host_barrier()
struct uint2 {
    unsigned x, y;
};
struct Dim3 {
    int x;
};
static Dim3 threadIdx, blockIdx, blockDim, gridDim;
static const void *host_kernel;
static void *host_lds;
static void host_barrier();
static void host_yield();
static float __uint_as_float(unsigned v)
{
    float f;
    std::memcpy(&f, &v, 4);
    return f;
}
static unsigned __float_as_uint(float f)
{
    unsigned v;
    std::memcpy(&v, &f, 4);
    return v;
}
static int atomicCAS(int *p, int want, int v)
{
    const int old = *p;
    if (old == want) *p = v;
    return old;
}

// vectors of N floats: aligned ones, and ones at any float's address
template <int N>
struct HostVecU;
template <int N>
struct alignas(4 * N) HostVec {
    float v[N];
    HostVec() = default;
    explicit HostVec(float x)
    {
        for (float &e : v) e = x;
    }
    HostVec(const HostVecU<N> &o) { std::memcpy(v, o.v, sizeof v); }
    float &operator[](int k) { return v[k]; }
    float operator[](int k) const { return v[k]; }
#define OP(o)                                                        \
    friend HostVec operator o(const HostVec &a, const HostVec &b)    \
    {                                                                \
        HostVec r;                                                   \
        for (int k = 0; k < N; ++k) r.v[k] = a.v[k] o b.v[k];        \
        return r;                                                    \
    }                                                                \
    friend HostVec operator o(const HostVec &a, float b) { return a o HostVec(b); } \
    friend HostVec operator o(float a, const HostVec &b) { return HostVec(a) o b; }
    OP(+) OP(-) OP(*)
#undef OP
};
template <int N>
struct HostVecU {
    float v[N];
    HostVecU() = default;
    HostVecU(const HostVec<N> &o) { std::memcpy(v, o.v, sizeof v); }
};

#include "resident_host.inc"  // dn_resident.inc, rewritten

using namespace dn;

// ---------------------------------------------------------------- threads
namespace {
constexpr size_t STACK = 512 * 1024;
struct Fiber {
    ucontext_t ctx;
    void *stack, *fake = nullptr;
    int block, thread;
    bool done = false, waiting = false;
};
ucontext_t sched;
const void *sched_stack;
size_t sched_size;
void *sched_fake;
Fiber *cur;
void (*kernel_entry)();

void leave(bool last)
{
    Fiber *f = cur;
    __sanitizer_start_switch_fiber(last ? nullptr : &f->fake, sched_stack, sched_size);
    swapcontext(&f->ctx, &sched);
    __sanitizer_finish_switch_fiber(f->fake, &sched_stack, &sched_size);
}
void start()
{
    __sanitizer_finish_switch_fiber(nullptr, &sched_stack, &sched_size);
    kernel_entry();
    cur->done = true;
    leave(true);
}

// advances the workgroups until all their threads have left
void run_grid(int blocks, int threads, size_t lds_bytes)
{
    static std::vector<void *> stacks;
    std::vector<std::unique_ptr<Fiber>> all;
    std::vector<char *> lds;
    for (int b = 0; b < blocks; ++b) {
        lds.push_back((char *)std::aligned_alloc(16, (lds_bytes + 15) / 16 * 16));
        std::memset(lds.back(), 0xff, lds_bytes);  // NaN
        __asan_poison_memory_region(lds.back() + lds_bytes, (lds_bytes + 15) / 16 * 16 - lds_bytes);
        for (int t = 0; t < threads; ++t) {
            auto f = std::make_unique<Fiber>();
            const size_t n = all.size();
            if (n == stacks.size())
                stacks.push_back(mmap(nullptr, STACK, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0));
            f->stack = stacks[n];
            f->block = b;
            f->thread = t;
            getcontext(&f->ctx);
            f->ctx.uc_stack.ss_sp = f->stack;
            f->ctx.uc_stack.ss_size = STACK;
            makecontext(&f->ctx, start, 0);
            all.push_back(std::move(f));
        }
    }
    blockDim.x = threads;
    gridDim.x = blocks;
    for (bool any = true; any;) {
        any = false;
        for (int b = 0; b < blocks; ++b) {
            bool open = true;  // all threads of the workgroup are at its barrier
            for (int t = 0; t < threads; ++t) {
                Fiber &f = *all[(size_t)b * threads + t];
                if (f.done || f.waiting) continue;
                any = true;
                cur = &f;
                threadIdx.x = t;
                blockIdx.x = b;
                host_lds = lds[b];
                __sanitizer_start_switch_fiber(&sched_fake, f.stack, STACK);
                swapcontext(&sched, &f.ctx);
                __sanitizer_finish_switch_fiber(sched_fake, nullptr, nullptr);
                open = open && (f.done || f.waiting);
            }
            if (!open) continue;
            for (int t = 0; t < threads; ++t) {
                Fiber &f = *all[(size_t)b * threads + t];
                if (f.waiting) any = true;
                f.waiting = false;
            }
        }
    }
    for (char *p : lds) {
        __asan_unpoison_memory_region(p, (lds_bytes + 15) / 16 * 16);
        std::free(p);
    }
}
}  // namespace
static void host_barrier()
{
    cur->waiting = true;
    leave(false);
}
static void host_yield() { leave(false); }

// ---------------------------------------------------------------- a run
namespace {
std::mt19937 rng;
float uni(float lo, float hi) { return lo + (hi - lo) * (float)(rng() >> 8) * 0x1p-24f; }

struct Grid {
    int nx, ny, fw, free_surf, nt, dtinv, points;
};
struct Point {
    int i, j, kind, idx;
};

// planes and arrays of their own size each, and what the kernel is told of them
struct Shot {
    Grid g;
    Layout lay;
    std::vector<std::unique_ptr<float[]>> mem;
    std::vector<std::pair<float *, size_t>> out;  // what a run leaves
    ResKernel k{};
    std::vector<std::unique_ptr<double[]>> dmem;
    std::vector<int> type;
    int nan_abort[2] = {0, 0};
    std::vector<Point> pts[2];
    float *arr(size_t n, float lo, float hi, bool result = false)
    {
        mem.emplace_back(new float[n]);
        for (size_t q = 0; q < n; ++q) mem.back()[q] = uni(lo, hi);
        if (result) out.push_back({mem.back().get(), n});
        return mem.back().get();
    }
    // a padded plane, zero outside the grid
    float *plane(float lo, float hi, int count = 1, bool result = false)
    {
        float *p = arr(lay.plane() * count, 0.0f, 0.0f, result);
        for (int c = 0; c < count; ++c)
            for (int j = 1; j <= g.ny; ++j)
                for (int i = 1; i <= g.nx; ++i) p[c * lay.plane() + lay.origin() + lay.off(j, i)] = uni(lo, hi);
        return p + lay.origin();
    }
    Shot(const Grid &gr) : g(gr)
    {
        rng.seed(7);
        lay.init(g.nx, g.ny);
        KArgs &a = k.a;
        a.nx = g.nx;
        a.ny = g.ny;
        a.pitch = lay.pitch;
        a.fw = g.fw;
        a.fw2 = 2 * g.fw;
        a.free_surf = g.free_surf;
        a.physics = CPH;
        a.mirror = g.free_surf && (CPH == 1 || CPH == 2);
        a.L = CL;
        a.nt_total = g.nt;
        a.dt = 0.003f;
        a.dh = 7.3f;
        a.dhi_el = a.dt / a.dh;
        a.dhi_vis = (float)(1.0 / a.dh);
        a.dthalbe = a.dt / 2.0f;
        for (int m = 0; m < 8; ++m) a.hc[m] = m == 0 ? 0.0f : (m % 2 ? 1.2f : -1.2f) / (float)(m * m);
        a.plane = (long)lay.plane();
        a.vx = plane(-1, 1, 1, true);
        a.vy = plane(-1, 1, 1, true);
        a.sxx = plane(-1, 1, 1, true);
        a.syy = CPH == 2 ? a.sxx : plane(-1, 1, 1, true);
        a.sxy = plane(-1, 1, 1, true);
        a.vxp1 = plane(-1, 1, 1, true);
        a.vyp1 = plane(-1, 1, 1, true);
        a.rip = plane(5, 20);
        a.rjp = plane(5, 20);
        a.muipjp = plane(0.1f, 0.3f);
        a.f = plane(0.1f, 0.3f);
        a.g = plane(0.4f, 0.6f);
        a.vmu = plane(10, 30);
        a.vpi = plane(60, 90);
        a.vmuij = plane(10, 30);
        for (auto &m : a.ani) m = plane(0.1f, 0.3f);
        a.tau_const = 1;
        a.ts0 = 0.05f;
        a.tp0 = 0.04f;
        a.tsij0 = 0.05f;
        for (int l = 0; l <= MAXL; ++l) {
            a.peta[l] = uni(1, 5);
            a.bip[l] = a.bjm[l] = uni(0.8f, 1);
            a.cip[l] = a.cjm[l] = uni(0.8f, 1);
            a.fs_bjm[l] = uni(0.8f, 1);
        }
        if (CL) {
            a.rmem = plane(-1, 1, CL, true);
            a.pmem = plane(-1, 1, CL, true);
            a.qmem = plane(-1, 1, CL, true);
        }
        a.fs_fjm = arr((size_t)g.nx + 1, 10, 30);
        a.fs_g = arr((size_t)g.nx + 1, 60, 90);
        a.fs_dme = arr((size_t)g.nx + 1, 0.1f, 1);
        a.vp = plane(2, 3);
        a.vs = plane(1, 2);
        a.rho = plane(1, 2);
        const size_t nxb = (size_t)g.ny * 2 * g.fw + 1, nyb = (size_t)2 * g.fw * g.nx + 1;
        for (float **p : {&a.psi_sxx_x, &a.psi_sxy_x, &a.psi_vxx, &a.psi_vyx, &a.psi_vxxs}) *p = arr(nxb, -0.1f, 0.1f, true);
        for (float **p : {&a.psi_syy_y, &a.psi_sxy_y, &a.psi_vyy, &a.psi_vxy}) *p = arr(nyb, -0.1f, 0.1f, true);
        for (const float **p : {&a.a_x, &a.a_xh, &a.a_y, &a.a_yh}) *p = arr((size_t)2 * g.fw + 1, -0.3f, 0.0f);
        for (const float **p : {&a.b_x, &a.b_xh, &a.b_y, &a.b_yh}) *p = arr((size_t)2 * g.fw + 1, 0.5f, 1.0f);
        // sources and receivers: the corners, and some cells inside
        std::vector<std::pair<int, int>> cells = {{1, 2}, {g.nx, 2}, {1, g.ny}, {g.nx, g.ny}, {g.nx / 2, g.ny / 2}};
        while ((int)cells.size() < g.points) cells.push_back({1 + (int)(rng() % g.nx), 2 + (int)(rng() % (g.ny - 1))});
        cells.resize((size_t)g.points);
        const int n = (int)cells.size();
        DevAcq &q = k.q;
        q.nsrc = q.ntr = n;
        q.nt = g.nt;
        q.signals = arr((size_t)n * g.nt, -1, 1);
        for (int c = 0; c < 3; ++c) q.adj[c] = arr((size_t)n * g.nt, -1, 1);
        for (int c = 0; c < 5; ++c) q.sec[c] = arr((size_t)n * g.nt, 0, 0, true);
        auto doubles = [&] {
            dmem.emplace_back(new double[n]);
            for (int t = 0; t < n; ++t) dmem.back()[t] = uni(0.1f, 1);
            return dmem.back().get();
        };
        q.src_sin = doubles();
        q.src_cos = doubles();
        q.rec_sqlam = doubles();
        q.rec_sqmu = doubles();
        for (int t = 0; t < n; ++t) type.push_back(CPH == 5 ? 1 : 1 + t % 4);
        q.src_type = type.data();
        q.nan_step = nan_abort;
        for (int t = 0; t < n; ++t) {
            const int i = cells[t].first, j = cells[t].second;
            if (CSW == 0) {
                pts[type[t] == 1 && CPH != 5].push_back({i, j, type[t] == 1 && CPH != 5 ? E_EXPLOSIVE : E_FORCE, t});
                pts[0].push_back({i, j, E_REC_V, t});
                if (CPH != 5) pts[1].push_back({i, j, E_REC_S, t});
            } else {
                pts[0].push_back({i, j, E_ADJ_FORCE, t});
                if (CPH != 5) pts[1].push_back({i, j, E_ADJ_P, t});
            }
        }
        StepCtl &c = k.c;
        c.seismo = CSW ? 0 : CPH == 2 ? 2 : CPH == 5 ? 1 : 4;
        c.probe = 1;
        c.quelltypb = CPH == 5 ? 1 : 7;
        c.invmat1 = 1;
        const size_t np = (size_t)g.nx * g.ny, slots = (size_t)((g.nt + g.dtinv - 1) / g.dtinv);
        for (float *&f : c.fwd) f = arr(np * slots, -1, 1, CSW == 0);
        c.wc = arr(np, -1, 1, true);
        c.wcu = arr(np, -1, 1, true);
        c.wcr = arr(np, -1, 1, true);
    }
    std::vector<float> results() const
    {
        std::vector<float> v;
        for (auto &o : out) v.insert(v.end(), o.first, o.first + o.second);
        v.push_back((float)nan_abort[0]);
        v.push_back((float)nan_abort[1]);
        return v;
    }
};

// steps 1..nt of the shot by a plan, in launches that end at `cut` and at nt
template <int RY, int VX>
void advance(Shot &s, const ResPlan &plan, int cut)
{
    ResPlan pl = plan;
    const int HP = 4 * ((CF + 3) / 4), LP = res_width(RY) + 2 * HP;
    // point lists by tile and owner thread
    std::vector<int> off[2], own[2];
    std::vector<uint2> ent[2];
    int most[2];
    for (int w = 0; w < 2; ++w) {
        struct E {
            int tile, own;
            uint2 e;
        };
        std::vector<E> v;
        for (const Point &q : s.pts[w]) {
            const int bx = (q.i - 1) / pl.tw, by = (q.j - 1) / pl.th, x = q.i - 1 - bx * pl.tw, y = q.j - 1 - by * pl.th;
            v.push_back({by * pl.gx + bx, y / RY * pl.nthx + x / VX,
                         {(unsigned)(q.kind << 24 | ((y + CF) * LP + HP + x)), (unsigned)q.idx}});
        }
        std::stable_sort(v.begin(), v.end(),
                         [](const E &a, const E &b) { return a.tile < b.tile || (a.tile == b.tile && a.own < b.own); });
        off[w].assign((size_t)pl.tiles() + 1, 0);
        for (const E &e : v) {
            off[w][(size_t)e.tile + 1]++;
            own[w].push_back(e.own);
            ent[w].push_back(e.e);
        }
        most[w] = *std::max_element(off[w].begin(), off[w].end());
        for (int t = 0; t < pl.tiles(); ++t) off[w][(size_t)t + 1] += off[w][t];
        own[w].push_back(0);
    }
    ResArgs &r = s.k.r;
    r = ResArgs{};
    r.tw = pl.tw;
    r.th = pl.th;
    r.gx = pl.gx;
    r.gy = pl.gy;
    r.nthx = pl.nthx;
    r.ncomp = pl.ncomp;
    r.nk_s = pl.nk_s;
    r.nk_v = pl.nk_v;
    r.cap = pl.cap;
    r.ncx = pl.ncx;
    r.ncy = pl.ncy;
    r.nve = most[0];
    r.nse = most[1];
    r.nlast = s.g.nt;
    r.fwdstore = CSW == 0;
    r.dtinv = s.g.dtinv;
    r.vp1_form = 1;
    r.quit = 1 << 30;
    r.rdh = 1.0 / (double)s.k.a.dh;
    std::unique_ptr<res_word[]> box(new res_word[(size_t)pl.tiles() * 2 * pl.cap]());
    r.mbox = box.get();
    r.abort = s.nan_abort + 1;
    r.voff = off[0].data();
    r.vown = own[0].data();
    r.vent = ent[0].data();
    r.soff = off[1].data();
    r.sown = own[1].data();
    r.sent = ent[1].data();
    unsigned tag = 1;
    for (int n = 1; n <= s.g.nt; n = r.n1 + 1) {
        r.n0 = n;
        r.n1 = n <= cut ? std::min(cut, s.g.nt) : s.g.nt;
        r.tag0 = tag;
        tag += (unsigned)(r.n1 - r.n0 + 2);
        host_kernel = &s.k;
        kernel_entry = [] { k_resident<CF, RY, VX, res_width(RY), CPH, CL, CSW>(*(const ResKernel *)host_kernel); };
        run_grid(pl.tiles(), pl.nthr, pl.lds + (size_t)((most[0] + most[1] + 1) & ~1) * sizeof(uint2));
    }
}

long fails = 0, plans = 0;

template <int S>
void shape(const Grid &g, std::vector<float> &want)
{
    constexpr int RY = res_shapes[S][0], VX = res_shapes[S][1];
    dn_params p{};
    p.nx = g.nx;
    p.ny = g.ny;
    p.fw = g.fw;
    p.free_surf = g.free_surf;
    p.fdorder = 2 * CF;
    p.physics = CPH;
    p.L = CL;
    if constexpr (RY <= res_rows(CF, CPH, CL, CSW)) {
        const ResPlan least = res_least(p, 163840 - 2048, S);
        if (!least.ok) return;
        for (int more : {0, 5}) {
            ResPlan pl = more ? res_plan(p, least.tiles() + more, 163840 - 2048, S) : least;
            if (!pl.ok || (more && pl.tiles() == least.tiles())) continue;
            if (more) {  // the threads of a launch with larger workgroups
                pl.nthr = std::min(pl.nthr + 64, res_maxt(RY, VX, CF, CL));
                pl.nk_s = pl.nk_v = (pl.cap + pl.nthr - 1) / pl.nthr;
            }
            std::printf("order %d physics %d L %d %s %dx%d fw %d: %dx%d cells a thread, %dx%d tiles of %dx%d\n", 2 * CF, CPH, CL,
                        CSW ? "adjoint" : "forward", g.nx, g.ny, g.fw, RY, VX, pl.gx, pl.gy, pl.tw, pl.th);
            std::fflush(stdout);
            Shot s(g);
            advance<RY, VX>(s, pl, more ? 2 : g.nt);
            const std::vector<float> got = s.results();
            if (want.empty()) want = got;
            ++plans;
            if (got.size() != want.size() || std::memcmp(got.data(), want.data(), got.size() * sizeof(float))) {
                ++fails;
                std::printf("  differs\n");
            }
            for (float v : got)
                if (!(std::fabs(v) < 1e30f)) {
                    ++fails;
                    std::printf("  not finite\n");
                    break;
                }
        }
    }
}
}  // namespace

int main(int argc, char **argv)
{
    std::vector<Grid> grids = {{24, 22, 0, 1, 4, 1, 0}, {37, 26, 5, 0, 4, 2, 15}, {70, 31, 6, 1, 4, 3, 15}, {90, 41, 3, 0, 4, 2, 1}};
    if (argc > 8) grids = {{atoi(argv[2]), atoi(argv[3]), atoi(argv[4]), atoi(argv[5]), atoi(argv[6]), atoi(argv[7]), atoi(argv[8])}};
    const int only = argc > 1 ? atoi(argv[1]) : -1;
    for (const Grid &g : grids) {
        std::vector<float> want;
        if (only < 0 || only == 0) shape<0>(g, want);
        if (only < 0 || only == 1) shape<1>(g, want);
        if (only < 0 || only == 2) shape<2>(g, want);
        if (only < 0 || only == 3) shape<3>(g, want);
        if (only < 0 || only == 4) shape<4>(g, want);
    }
    std::printf("%s, %ld plans\n", fails ? "resident loop wrong" : "resident loop ok", plans);
    return fails || !plans ? 1 : 0;
}
