// Chip-resident time loop (dn_resident.inc): launch arguments and the pool of
// halo mailboxes.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "dn_resident_plan.h"

namespace dn {

typedef unsigned long long res_word;

struct ResArgs {
    int tw, th, gx, gy, nthx, ncomp, nk_s, nk_v, cap, ncx, ncy, nve, nse;
    int n0, n1, nlast;  // time steps of this launch, last step of the run
    int fwdstore, dtinv, vp1_form;
    int quit;           // last step before the first tile abandons the run (dn_set_loop)
    double rdh;         // 1 / DH
    unsigned tag0;
    res_word *mbox;
    int *abort;
    // sources and receivers per tile, sorted by owner thread:
    // {kind << 24 | LDS element, index}
    const int *voff, *vown, *soff, *sown;
    const uint2 *vent, *sent;
};

// the point lists of a plan, one block: per list offsets, owners, entries
struct ResPoints {
    std::vector<int> blk;
    size_t off[4] = {}, own[4] = {}, ent[4] = {};  // positions in it (ints)
    bool ok[4] = {};   // no point that the loop has no place for
    int most[4] = {};  // entries of a tile, at most
};

// one workgroup of a launch that holds several shots
struct ResBlock {
    int shot, tile;
};

// the kernel's one argument: a shot, or the shots of the launch (tab) and
// the shot and tile of every workgroup (blk)
struct ResKernel {
    KArgs a;
    StepCtl c;
    DevAcq q;
    ResArgs r;
    const ResKernel *tab;
    const ResBlock *blk;
};

// is there a compiled kernel for this run (sw 0 forward, 1 adjoint) with ry rows per thread
bool res_compiled(int fdoh, int physics, int L, int sw, int ry);
// enqueue one launch of as many workgroups, with the threads, LDS and thread
// shape of pl on a device with lds_max bytes of LDS per workgroup; false when
// the runtime refuses it
bool res_launch(const ResKernel &k, const ResPlan &pl, int blocks, int fdoh, int sw, size_t lds_max, void *stream);

// The mailboxes of a device: one allocation shared by the contexts on it,
// made with the first and given back with the last, and the account of its
// CUs.  A run takes a range of mailboxes and as many CUs as it has tiles for
// its duration; runs that find too few take the sweeps instead of waiting,
// so runs of several threads and streams never wait for each other's CUs.
// Step tags only grow, so a word left by an earlier run matches no later
// tag.  Thread-safe.
struct ResPool;
ResPool *res_pool_open(int device);  // nullptr: no pool (no memory)
void res_pool_close(ResPool *p);
int res_pool_cus(const ResPool *p);
size_t res_pool_lds(const ResPool *p);
// step tags of a run: one for each step and two for each launch
constexpr unsigned res_tags(int steps) { return (unsigned)steps + 2u * (unsigned)(steps / RES_CHUNK + 2); }
struct ResLease {
    res_word *mbox = nullptr;
    unsigned tag0 = 0;
};
// mailboxes of so many words, CUs for so many tiles, and step tags
bool res_pool_take(ResPool *p, int tiles, size_t words, unsigned tags, ResLease *out);
void res_pool_give(ResPool *p, const ResLease &l);

}  // namespace dn
