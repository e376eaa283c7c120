// Host side of the chip-resident time loop: the pool of mailboxes and CUs of a device, and the dispatch to the compiled kernels.
#include "dn_resident.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <new>
#include <vector>

namespace dn {

template <int F, int GROUP>
bool res_launch_f(const ResKernel &k, const ResPlan &pl, int blocks, int sw, size_t lds_max, hipStream_t s);

bool res_launch(const ResKernel &k, const ResPlan &pl, int blocks, int fdoh, int sw, size_t lds_max, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
#define DN_F(F)                                                                \
    case F:                                                                    \
        return k.a.physics != 1 ? res_launch_f<F, 1>(k, pl, blocks, sw, lds_max, s) \
               : k.a.L > 0      ? res_launch_f<F, 2>(k, pl, blocks, sw, lds_max, s) \
                                : res_launch_f<F, 0>(k, pl, blocks, sw, lds_max, s);
    switch (fdoh) {
        DN_F(1) DN_F(2) DN_F(3) DN_F(4) DN_F(5) DN_F(6)
    }
#undef DN_F
    return false;
}

bool res_compiled(int fdoh, int physics, int L, int sw, int ry)
{
    return physics >= 1 && physics <= 5 && (L == 0 || (physics == 1 && L <= 3)) && ry <= res_rows(fdoh, physics, L, sw);
}

// ---------------------------------------------------------------- the pool
struct ResPool {
    struct Range {
        size_t at, words;
        int tiles;
    };
    std::mutex m;
    int device = 0, refs = 0, ncu = 0, tiles = 0;
    size_t lds = 0, words = 0;
    res_word *mem = nullptr;
    unsigned next = 1;
    std::vector<Range> busy;  // by position
};

namespace {
std::mutex pools_m;
std::map<int, ResPool *> pools;

// tags start at 1: no word of zeros matches one
bool clear(ResPool *p)
{
    hipStream_t s = nullptr;
    const bool ok = hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess &&
                    hipMemsetAsync(p->mem, 0, p->words * sizeof(res_word), s) == hipSuccess &&
                    hipStreamSynchronize(s) == hipSuccess;
    if (s) (void)hipStreamDestroy(s);
    if (ok)
        p->next = 1;
    else
        (void)hipGetLastError();
    return ok;
}
}  // namespace

ResPool *res_pool_open(int device)
{
    std::lock_guard<std::mutex> g(pools_m);
    ResPool *&p = pools[device];
    if (p) {
        ++p->refs;
        return p;
    }
    ResPool *q = new (std::nothrow) ResPool();
    if (!q) return nullptr;
    int ncu = 0, lds = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess) {
        (void)hipGetLastError();
        delete q;
        return nullptr;
    }
    q->device = device;
    q->ncu = ncu;
    q->lds = (size_t)lds;
    q->words = (size_t)ncu * 2 * RES_CAP;
    if (hipMalloc((void **)&q->mem, q->words * sizeof(res_word)) != hipSuccess || !clear(q)) {
        (void)hipGetLastError();
        if (q->mem) (void)hipFree(q->mem);
        delete q;
        return nullptr;
    }
    q->refs = 1;
    p = q;
    return q;
}

void res_pool_close(ResPool *p)
{
    if (!p) return;
    std::lock_guard<std::mutex> g(pools_m);
    if (--p->refs > 0) return;
    pools.erase(p->device);
    (void)hipFree(p->mem);
    delete p;
}

int res_pool_cus(const ResPool *p) { return p->ncu; }
size_t res_pool_lds(const ResPool *p) { return p->lds; }

bool res_pool_take(ResPool *p, int tiles, size_t words, unsigned tags, ResLease *out)
{
    std::lock_guard<std::mutex> g(p->m);
    if (p->tiles + tiles > p->ncu) return false;
    size_t at = 0, k = 0;
    for (; k < p->busy.size(); ++k) {  // first gap
        if (p->busy[k].at - at >= words) break;
        at = p->busy[k].at + p->busy[k].words;
    }
    if (at + words > p->words) return false;
    // tags must not come round again over words that hold them: an idle pool
    // half way through them starts afresh
    if (p->busy.empty() && p->next > 0x80000000u && !clear(p)) return false;
    if (tags > 0x7fffffffu || p->next > 0xffffffffu - tags) return false;
    out->mbox = p->mem + at;
    out->tag0 = p->next;
    p->next += tags;
    p->busy.insert(p->busy.begin() + (long)k, ResPool::Range{at, words, tiles});
    p->tiles += tiles;
    return true;
}

void res_pool_give(ResPool *p, const ResLease &l)
{
    std::lock_guard<std::mutex> g(p->m);
    for (size_t k = 0; k < p->busy.size(); ++k)
        if (p->mem + p->busy[k].at == l.mbox) {
            p->tiles -= p->busy[k].tiles;
            p->busy.erase(p->busy.begin() + (long)k);
            return;
        }
}

}  // namespace dn
