// Persistent batched scan: one launch walks the tiles of many scans (datasets
// of uneven N and M, and several phenotypes per dataset).
//
// The host keeps one work list per tile kind (FAST, GENERAL, SPARSE) for the scans that go through the screen
// and one for the others, each run by its
// own kernel (persistent, but for the screen's) so that a kernel holds the registers of one tile kind
// only. It orders the items of a list so that consecutive items share SNP data
// (tile-major, phenotype-minor) and cuts the list into NQ contiguous queues of
// equal estimated cost, one per XCD. A workgroup pulls items from the queue of
// its XCD (workgroups are dealt to XCDs round-robin, so blockIdx % 8 is its
// XCD), one item ahead so that the atomic overlaps the current tile, and, when
// that queue is empty, from the others in turn. Every pull is one atomicAdd; a
// claimed slot below its queue's end is always processed, and a pull past the
// end of every queue ends the workgroup, so all workgroups exit once the items
// run out. The queue heads are reset by a
// kernel (not a memset) so that the reset and the scan can be captured in one
// hipGraph and replayed.
#pragma once

#include "kern_mfma.h"
#include "kern_plain.h"
#include "kern_screen.h"

namespace epi {

constexpr int NQ = 8;     // work queues, one per XCD
constexpr int NKIND = 3;  // tile kinds: 0 FAST, 1 GENERAL, 2 SPARSE
constexpr int NLIST = 2 * NKIND;  // work lists: the kinds of the screened scans, then of the others

struct BatchArgs {
    const MfmaScan *mscan;   // [nscan]
    const PlainScan *pscan;  // [nscan]
    const int4 *work;        // {a0, b0, alen | blen << 8 | general << 16, scan}
    int *qpos;               // [NQ] next item of each queue of this kernel's list (reset to qbegin)
    const int *qend;         // [NQ] one past the last item of each queue
    HitSink hs;
};

struct ScreenBatchArgs {
    const MfmaScan *mscan;   // [nscan]
    const ScreenCut *cut;    // [nscan]
    const int4 *work;        // the launch's items, as in BatchArgs
    int nitems;
    int item0;               // index of work[0] in the kind's list
    CandSink cs;
};

// The hit counter and, behind it, the screen's: candidates and blocks to redo of each tile kind, and the
// candidates of lists that were emptied.
struct Counters {
    unsigned long long nhits;
    uint32_t screen[2 * NKIND];
    unsigned long long emptied;
};

// Clears words [from, n) of p, the counters of a scan, and m words of q, the masks of the blocks of a new tile list, in one
// small launch. (As two hipMemsetAsync calls N = 500, M = 2000, 94 us a scan, took 2.6 us more, and 45 us more with a new
// list; a second launch for the masks costs a first scan 30 us.)
__global__ __launch_bounds__(256) void clear_words(uint32_t *p, uint32_t from, uint32_t n, uint32_t *q, size_t m)
{
    const size_t i = blockIdx.x * 256ull + threadIdx.x;
    if (i >= from && i < n) p[i] = 0u;
    if (i < m) q[i] = 0u;
}

// Queue heads of every list ([NLIST][NQ]) and the counters.
__global__ void batch_reset(int *qpos, const int *qbegin, Counters *n)
{
    const int t = threadIdx.x;
    if (t < NLIST * NQ) qpos[t] = qbegin[t];
    if (t < 2 * NKIND) n->screen[t] = 0u;
    if (t == 0) n->nhits = n->emptied = 0ull;
}

// Called by one thread: the next item for a workgroup whose home queue is
// `home`, or -1 when every queue is exhausted.
__device__ __forceinline__ int next_item(const BatchArgs &B, int home)
{
    for (int k = 0; k < NQ; k++) {
        const int q = (home + k) % NQ;
        if (__hip_atomic_load(&B.qpos[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= B.qend[q]) continue;
        const int v = atomicAdd(&B.qpos[q], 1);
        if (v < B.qend[q]) return v;
    }
    return -1;
}

// Threads of a workgroup of the batch kernel for tile kind KIND: the tile's own
// (FAST 4 TA, one wave per SIMD; GENERAL and SPARSE 8 TA).
template <int TA, int KIND>
constexpr int batch_threads() { return KIND == 0 ? fast_threads<TA>() : KIND == 1 ? general_threads<TA>() : sparse_threads<TA>(); }
template <int TA, int KIND>
constexpr int batch_waves_per_simd() { return KIND == 0 ? fast_waves_per_simd<TA>() : 64 / TA; }

// TA: FAST and SPARSE tiles are TA x 64 (TA = 32 or 64), GENERAL tiles
// TA x 32. KIND: the list this kernel runs (0 FAST, 1 GENERAL, 2 SPARSE).
template <int TA, int KIND>
__global__ __launch_bounds__((batch_threads<TA, KIND>()), (batch_waves_per_simd<TA, KIND>())) void mfma_batch_kernel(
    const BatchArgs B)
{
    constexpr int GA = TA;
    constexpr int LDS = KIND == 1 ? general_lds<GA>() : KIND == 2 ? sparse_lds<TA>() : fast_lds<TA>();
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];
    __shared__ int item;
    __shared__ int4 wsh;
    const int home = blockIdx.x % NQ;
    const DumpSink nodump = {};
    // Thread 0 claims the next slot of the home queue one item ahead, so the
    // atomic's latency overlaps the current tile.
    int pend = 0;
    if (threadIdx.x == 0) pend = atomicAdd(&B.qpos[home], 1);
    for (;;) {
        __syncthreads();  // the previous tile is done with LDS and the shared item
        if (threadIdx.x == 0) {
            const int it = pend < B.qend[home] ? pend : next_item(B, home);
            item = it;
            if (it >= 0) {
                wsh = B.work[it];
                if (pend < B.qend[home]) pend = atomicAdd(&B.qpos[home], 1);
            }
        }
        __syncthreads();
        const int it = item;
        if (it < 0) break;
        const int4 w = wsh;
        const int a0 = __builtin_amdgcn_readfirstlane(w.x), b0 = __builtin_amdgcn_readfirstlane(w.y);
        const int ext = __builtin_amdgcn_readfirstlane(w.z), sc = __builtin_amdgcn_readfirstlane(w.w);
        // the scan's descriptor stays in memory (its fields load where used)
        // rather than held in registers across the tile
        const MfmaScan &S = B.mscan[sc];
        HitSink hs = B.hs;
        hs.tag = sc;
        const int a1 = a0 + (ext & 255), b1 = b0 + ((ext >> 8) & 255);
        if (KIND == 1)
            mfma_general_tile<GA, false>(S, hs, nodump, a0, a1, b0, b1, lds);
        else if (KIND == 2)
            mfma_sparse_tile<TA, false>(S, hs, nodump, a0, a1, b0, b1, lds);
        else
            mfma_fast_tile<TA, false>(S, hs, nodump, a0, a1, b0, b1, lds);
    }
}

// A list through the screen: one workgroup per item (two per SPARSE item), in the order of the list, with the XCD
// mapping of single scans (a persistent grid that pulls from the queues measured 5 % more at N = 4000, M = 20000).
// NC (screen_gen_tile) is one for the list: both
// variants in one kernel cost 1.5 % at N = 2504.
template <int TA, int KIND, bool NC = false>
__global__ __launch_bounds__(scr_threads<TA>(), 2) void screen_batch_kernel(const ScreenBatchArgs B)
{
    constexpr int HALVES = KIND == 2 ? 2 : 1, NBLK = scr_blocks(TA, KIND == 1 ? 32 : 64, KIND != 0);
    __shared__ __attribute__((aligned(16))) uint32_t wl[SCR_GEN_ROWS * sw_row<2>()];
    __shared__ float4 mg[KIND ? 2 * (TA + 32) : TA + 64];
    __shared__ float2 mg2[TA];
    const int t = xcd_tile(blockIdx.x, B.nitems * HALVES), it = t / HALVES;
    const int4 w = B.work[it];
    const int a0 = __builtin_amdgcn_readfirstlane(w.x), ext = __builtin_amdgcn_readfirstlane(w.z);
    const int sc = __builtin_amdgcn_readfirstlane(w.w), a1 = a0 + (ext & 255);
    int b0 = __builtin_amdgcn_readfirstlane(w.y), b1 = b0 + ((ext >> 8) & 255);
    // by value: the descriptors' fields would otherwise be loaded again wherever a store may alias them
    // (N = 4000, M = 20000 with 1 % missing calls: 9.1 against 7.2 ms a phenotype)
    const MfmaScan S = B.mscan[sc];
    const ScreenCut C = B.cut[sc];
    uint32_t block0 = (uint32_t)(B.item0 + it) * NBLK;
    if constexpr (KIND == 0) {
        if (C.nd == 1)
            screen_fast_tile<TA, 1>(S, C, B.cs, a0, a1, b0, b1, block0, wl, mg, mg2);
        else
            screen_fast_tile<TA, 2>(S, C, B.cs, a0, a1, b0, b1, block0, wl, mg, mg2);
    } else {
        if (!scr_half<TA>(t % HALVES, HALVES, (uint32_t)(B.item0 + it), b0, b1, block0)) return;
        if (C.nd == 1)
            screen_gen_tile<TA, 1, NC>(S, C, B.cs, a0, a1, b0, b1, block0, wl, mg);
        else
            screen_gen_tile<TA, 2, NC>(S, C, B.cs, a0, a1, b0, b1, block0, wl, mg);
    }
}

// NT: FAST tiles are NT/16 x 64 (NT = 512 or 256); GENERAL tiles are 16 x 64.
template <int NT, int GEN>
__global__ __launch_bounds__(NT, GEN ? 2 : 4) void plain_batch_kernel(const BatchArgs B)
{
    __shared__ PlainLds<!GEN> lds;
    __shared__ int item;
    __shared__ int4 wsh;
    const int home = blockIdx.x % NQ;
    const DumpSink nodump = {};
    int pend = 0;
    if (threadIdx.x == 0) pend = atomicAdd(&B.qpos[home], 1);
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) {
            const int it = pend < B.qend[home] ? pend : next_item(B, home);
            item = it;
            if (it >= 0) {
                wsh = B.work[it];
                if (pend < B.qend[home]) pend = atomicAdd(&B.qpos[home], 1);
            }
        }
        __syncthreads();
        const int it = item;
        if (it < 0) break;
        const int4 w = wsh;
        const int a0 = __builtin_amdgcn_readfirstlane(w.x), b0 = __builtin_amdgcn_readfirstlane(w.y);
        const int ext = __builtin_amdgcn_readfirstlane(w.z), sc = __builtin_amdgcn_readfirstlane(w.w);
        const PlainScan S = B.pscan[sc];
        HitSink hs = B.hs;
        hs.tag = sc;
        const int a1 = a0 + (ext & 255), b1 = b0 + ((ext >> 8) & 255);
        if constexpr (GEN)
            plain_tile<256, false, false>(S, hs, nodump, a0, a1, b0, b1, lds);
        else
            plain_tile<NT, true, false>(S, hs, nodump, a0, a1, b0, b1, lds);
    }
}

}  // namespace epi
