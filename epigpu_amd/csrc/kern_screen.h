// Screened pair scan (gfx950, v_mfma_f32_32x32x64_f8f6f4 on 6-bit operands).
//
// Almost no pair of a scan is a hit, so most pairs need no exact table: a bound
// on their statistics settles them. The screen kernels contract the class
// masks with a coarse phenotype v instead of the 24-bit q of kern_mfma.h, keep
// every pair whose true statistics could pass the thresholds (candidates),
// and resolve_kernel computes the candidates' tables exactly, as integers, and
// decides them in FP64 with the same code as the exact tiles. The hits and
// their values are those of exact tiles of the same height.
// What decides which pairs are dropped has fewer bits than a table: 6-bit digits, FP32 sums and an
// FP32 decision. The bound below pays for the digits, every sum is an exact integer (screen_dump shows them), and the thresholds'
// margin covers the decision.
//
// Coarse phenotype: v = D0, or v = 32 D1 + D0, with digits representable in FP6 (E2M3:
// in units of 1/8 the integers 0..16, then steps of 2 to 30 and of 4 to 60),
// |v| <= 60 or 1980; q ~ delta v + offset by least squares, and r is the rest. The
// rate of 6-bit MFMA operands is twice that of 8-bit ones, and a
// count and one or two digits replace the count and three limbs: 8 or 12 instead of 16 MACs
// per pair and individual without missing calls, at twice the rate.
//
// The class masks are those of an SNP's two rarest classes (rbits), and of the commonest where it is needed: the
// statistics do not depend on the classes' names, and the sparser the masks, the less power the
// MFMAs draw. A register-only loop runs 8.8 POP/s at 33 % ones, 9.1 at 22 %, 9.9 at 10 % (the clock falls to
// about 1.8 GHz in the scans).
//
// What bounds it: the matrix cores and their power. At N = 8000, M = 50000 without missing calls a scan's
// kernels take 34.5 ms (exact 64 x 64 tiles: 92-97 ms): 2.4e14 operations at 7.0 POP/s, against the 8.0 POP/s that
// a register-only loop of this MFMA with five VALU instructions beside each sustains (9.1 without any,
// 4.8 for v_mfma_i32_32x32x32_i8); the matrix cores are busy 81 % of the cycles, at 1.8 GHz.
//
// Bound: over a pair's complete cases let P y be the projection of a phenotype
// onto the cell-constant vectors less the mean, so SSB(y) = |P y|^2. Then
//     |P q| <= delta |P v| + |P r| <= delta |P v| + eps,   eps = |r|,
// and likewise sqrt(SSI(q)) <= delta sqrt(SSI(v)) + eps, since SSI(y) = |A y|^2 with A
// linear and SSI <= SSB <= |y|^2 for every y. With SST the total sum of squares,
//     F > t1   <=>  SSB > k1 SST,  k1 = t1 d1 / (d2 + t1 d1)
//     F2 > t2  =>   SSI > (4 t2 / d2) (SST - SSB), and since SSB >= SSI also
//                   SSB > k2 SST,  k2 = 4 t2 / (d2 + 4 t2).
// A pair is a candidate unless these fail with SSB, SSI replaced by their upper
// bounds and the thresholds lowered by 2 % (the margin of the exact tiles'
// FP32 screen, far above the rounding of the FP32 sums here: counts and
// digit sums are exact integers below 2^24).
#pragma once

#include "kern_mfma.h"
#include "screen_rules.h"

namespace epi {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Dwords per 32 individuals of the weights of ND digits: codes of D0 (6), of D1 (6), phenotype present, pad.
template <int ND>
constexpr int sw_row() { return 8 * ND; }
constexpr int SCR_WIN = 512; // words (of 32 individuals) of weights in LDS at a time
constexpr int SCR_LDS_ROWS = SCR_WIN + 2;  // the pipeline reads one step past the window
constexpr int SCR_GEN_ROWS = SCR_WIN + 4;
template <int TA>
constexpr int scr_threads() { return 64 * TA / SCR_A; }  // a workgroup takes a tile of TA = 32 or 64 a-SNPs
constexpr int SCR_REDO = 8;   // candidates per pair slot of a wave (64 pairs) above which the exact tile redoes its pairs

// Per SNP and phenotype: counts and sums of v (one and two digits) of the two rarest classes and
// the commonest one (present phenotypes; the fourth sum is padding), divided by 64 as the kernels' accumulators are, and
// the sum of z over all calls.
struct ScrMarg {
    float n[3], zs;
    float s[2][4];
};

// The cut of one scan (thresholds and phenotype), in units of v / 8 (sums of squares / 64).
struct ScreenCut {
    float N;              // complete cases / 64
    float thr0, slope2;   // level 0: sum s^2 / n > thr0 + 2 nfac slope2
    float eps;            // |r| / (8 delta)
    float sst;            // SST(q) / (64 delta^2)
    float nv;             // complete cases
    // GENERAL tiles: nv and N bound the pairs' complete cases from above
    float vs;             // sum of v over the phenotypes present / 64
    float zunit, zall;    // sums of squares per unit of z (from below); sum of z over all individuals
    float kap0, kslope2;  // level 0: sum s^2 / n > (kap0 + 2 nfac kslope2) SST - kroot
    float kroot, c0;      // c0: q ~ delta (v + c0), scaled as v is
    float t1s, t2s;       // lowered thresholds
    int test, safe;
    int nd;               // digits of v; 0: the scan is not screened
    float rate;           // predicted candidates per pair of unrelated SNPs
};

struct CandSink {
    int4 *cand;               // {a, b, scan, 0}; a == b: void
    uint32_t *count;          // [0] candidates, [1] blocks to redo
    uint32_t cap;
    uint32_t *redo;           // blocks (scr_blocks) to redo
    uint32_t *mask;           // per block, 0 between scans: bit w: the rows SCR_A w on of the block are to be redone
};

// The sums of the screen for every pair of a rectangle, a > b, instead of its decisions (epi_screen_dump).
struct ScreenDump {
    float *n, *s;             // [pair][9] counts and sums of v, both / 64, in genotype order
    int a0, b0, nb;
};

struct ScreenArgs {
    MfmaScan S;
    ScreenCut cut;
    CandSink cs;
    const int4 *tiles;
    int ntiles;
    int tile0;                // index of tiles[0] in the scan's list
    int halves;               // GENERAL kernel: workgroups per tile (1: 32 b, 2: SPARSE tiles of 64 b)
};

// The FP6 image of 32 individuals in a lane: element s occupies bits 6s..6s+5 of
// 192. Individual k (bit k of a bitplane word) goes to the element whose lowest
// bit is at bit k of a dword: even k in the first 96 bits, odd k (after a
// shift by one) in the last 96. The lowest bits of the elements at these
// positions are three masks of the word, and element s = scr_slot(k).
constexpr uint32_t SP0 = 0x41041041u, SP1 = 0x10410410u, SP2 = 0x04104104u;

__host__ __device__ constexpr int scr_slot(int k)
{
    const int e = k & ~1;  // bit position in the (shifted) word
    for (int s = 0; s < 16; s++)
        if (6 * s % 32 == e) return s + (k & 1 ? 16 : 0);
    return -1;
}

struct Fp6 {
    uint32_t d[6];
};

// 0/1 elements (0 or 0.125) of a bitplane word: seven VALU instructions.
__device__ __forceinline__ Fp6 scr_spread(uint32_t x)
{
    const uint32_t y = x >> 1;
    return {{x & SP0, x & SP1, x & SP2, y & SP0, y & SP1, y & SP2}};
}

// All six bits of every element set: (T << 6) - T over each 96-bit half.
__device__ __forceinline__ Fp6 scr_fill(const Fp6 &t)
{
    Fp6 m;
#pragma unroll
    for (int h = 0; h < 6; h += 3) {
        const uint32_t t0 = t.d[h], t1 = t.d[h + 1], t2 = t.d[h + 2];
        unsigned c0, c1, c2;
        m.d[h] = __builtin_subc(t0 << 6, t0, 0u, &c0);
        m.d[h + 1] = __builtin_subc(__builtin_amdgcn_alignbit(t1, t0, 26), t1, c0, &c1);
        m.d[h + 2] = __builtin_subc(__builtin_amdgcn_alignbit(t2, t1, 26), t2, c1, &c2);
    }
    return m;
}

__device__ __forceinline__ v8i scr_op(const Fp6 &f)
{
    return (v8i){(int)f.d[0], (int)f.d[1], (int)f.d[2], (int)f.d[3], (int)f.d[4], (int)f.d[5], 0, 0};
}

// FP6 x FP6 MFMA, plain and with the A operand scaled by 32 (E8M0 exponent 132).
__device__ __forceinline__ v16f scr_mfma(const v8i &a, const v8i &b, const v16f &c)
{
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 2, 2, 0, 0, 0, 0);
}
__device__ __forceinline__ v16f scr_mfma32(const v8i &a, const v8i &b, const v16f &c)
{
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 2, 2, 0, 0x84848484, 0, 0x7f7f7f7f);
}

// Twice the number of occupied cells: a count is 0 or a float whose bits exceed 2 (min and three-operand adds;
// a minimum with 1 would be rewritten as nine compares).
__device__ __forceinline__ float scr_nfac2(const float n[9])
{
    uint32_t o[9];
#pragma unroll
    for (int c = 0; c < 9; c++) o[c] = __float_as_uint(n[c]) < 2u ? __float_as_uint(n[c]) : 2u;
    return (float)(int)((o[0] + o[1] + o[2]) + (o[3] + o[4] + o[5]) + (o[6] + o[7] + o[8]));
}

// 1/n from above: the exponent of n negated and its mantissa mirrored, between
// 1/n and 1.125/n (the linear bound 1 - f/2 >= 1/(1+f) on 0 <= f <= 1), huge for n = 0.
__device__ __forceinline__ float rcp_above(float n) { return __uint_as_float(0x7F000000u - __float_as_uint(n)); }

// Second stage of the screen, per lane: the bounds above in FP32, from the
// nine cells' counts n and sums s (both / 64). SST is that of the pair's
// complete cases from below, sst, and nc their count.
__device__ __forceinline__ bool screen_bound(const float n[9], const float s[9], float nc, float sst, const ScreenCut &C)
{
    float nfac = 0.0f, N = 0.0f, T = 0.0f, m[9], q = 0.0f;
#pragma unroll
    for (int c = 0; c < 9; c++) {
        const bool occ = n[c] > 0.0f;
        nfac += occ ? 1.0f : 0.0f;
        N += n[c];
        T += s[c];
        m[c] = occ ? s[c] * __builtin_amdgcn_rcpf(n[c]) : 0.0f;
        q += occ ? m[c] * s[c] : 0.0f;
    }
    const float d1 = nfac - 1.0f, d2 = nc - nfac;
    if (!(d1 >= 1.0f) || !(d2 >= 1.0f)) return false;
    if (C.test != 'f' && !C.safe && !(nfac > 6.0f)) return false;
    const float mbar = T * __builtin_amdgcn_rcpf(N);
    const float ssb = fmaxf(q - T * mbar, 0.0f);
    const float rb = sqrtf(ssb) * 1.0001f + C.eps, ub = rb * rb;  // SSB(q) from above
    const float k1 = C.t1s * d1;
    if (ub * (d2 + k1) > k1 * sst) return true;
    if (C.test == 'f') return false;
    const float ssw = sst - ub;
    if (!(ub * d2 > 4.0f * C.t2s * ssw)) return false;  // SSI <= SSB
    float R[3], Cm[3];
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const float nr = n[3 * r] + n[3 * r + 1] + n[3 * r + 2], nk = n[r] + n[r + 3] + n[r + 6];
        R[r] = nr > 0.0f ? (s[3 * r] + s[3 * r + 1] + s[3 * r + 2]) * __builtin_amdgcn_rcpf(nr) : 0.0f;
        Cm[r] = nk > 0.0f ? (s[r] + s[r + 3] + s[r + 6]) * __builtin_amdgcn_rcpf(nk) : 0.0f;
    }
    float ssi = 0.0f;
#pragma unroll
    for (int c = 0; c < 9; c++) {
        const float t = m[c] - R[c / 3] - Cm[c % 3] + mbar;
        ssi += n[c] > 0.0f ? n[c] * t * t : 0.0f;
    }
    const float ri = sqrtf(ssi) * 1.0001f + C.eps;
    return ri * ri * d2 > 4.0f * C.t2s * ssw;
}

__device__ __forceinline__ void screen_dump(const ScreenDump &D, const MfmaScan &S, int a, int b, const float n[9], const float s[9])
{
    const size_t p = (size_t)(a - D.a0) * D.nb + (b - D.b0);
    const int ca = S.marg[a].cls, cb = S.marg[b].cls;
#pragma unroll
    for (int c = 0; c < 9; c++) {
        const int o = 3 * ((ca >> (2 * (c / 3))) & 3) + ((cb >> (2 * (c % 3))) & 3);
        D.n[9 * p + o] = n[c];
        D.s[9 * p + o] = s[c];
    }
}

// n rows of weights from global memory into LDS, four loads in flight per thread.
template <int NT, int ROW>
__device__ __forceinline__ void scr_stage(uint32_t *wl, const uint32_t *src, int n, int tid)
{
    const int last = n * (ROW / 4) - 1;  // threads past the end move the last piece
    const uint4 *g = reinterpret_cast<const uint4 *>(src);
    uint4 *l = reinterpret_cast<uint4 *>(wl);
    for (int i = tid; i <= last; i += 4 * NT) {
        const int i1 = i + NT < last ? i + NT : last, i2 = i + 2 * NT < last ? i + 2 * NT : last,
                  i3 = i + 3 * NT < last ? i + 3 * NT : last;
        const uint4 v0 = g[i], v1 = g[i1], v2 = g[i2], v3 = g[i3];
        l[i] = v0;
        l[i1] = v1;
        l[i2] = v2;
        l[i3] = v3;
    }
}

// A wave's candidates into the list, or its half of a block into the redo list: bit k of
// bits is the lane's pair (a(k), b(k)); wave wid of the tile or half whose first block is block0. Every lane calls.
template <int NB, class Pair>
__device__ __forceinline__ void scr_append(const CandSink &cs, uint32_t bits, uint32_t block0, int wid, int scan, Pair pair)
{
    if (__ballot(bits != 0u) == 0ull) return;
    uint32_t total = 0;
#pragma unroll
    for (int k = 0; k < NB; k++) total += __popcll(__ballot((bits >> k) & 1u));
    const int lane = __lane_id();
    uint32_t base = 0;
    if (lane == 0 && total <= SCR_REDO * NB) base = atomicAdd(cs.count, total);
    base = __builtin_amdgcn_readfirstlane(base);
    if (total > SCR_REDO * NB || base > cs.cap || total > cs.cap - base) {
        // too many for the list: the exact tile redoes the wave's pairs. Slots already reserved are voided.
        if (total <= SCR_REDO * NB)
            for (uint32_t i = base + lane; i < cs.cap && i < base + total; i += 64) cs.cand[i] = make_int4(0, 0, 0, 0);
        if (lane == 0) {
            const uint32_t block = block0 + (wid >> 1);
            if (atomicOr(&cs.mask[block], 1u << (wid & 1)) == 0u) cs.redo[atomicAdd(cs.count + 1, 1u)] = block;
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < NB; k++) {
        const uint64_t mask = __ballot((bits >> k) & 1u);
        if ((bits >> k) & 1u) {
            int a, b;
            pair(k, a, b);
            cs.cand[base + __popcll(mask & ((1ull << lane) - 1ull))] = make_int4(a, b, scan, 0);
        }
        base += __popcll(mask);
    }
}

// ---------------------------------------------------------------- FAST ----
// Tile TA a x 64 b without missing calls. Each wave owns 16 a x 64 b: 32 A rows
// (a, g) for classes g in {0, 1}, row m = 2 a + g, times three weights (the
// mask itself for the count, and the mask AND the codes of D0 and D1), against
// four B blocks of 32 b (class h of b-SNPs 32 bg + m): 12 MFMAs per 64
// individuals. D1 accumulates into the accumulators of D0 with the MFMA's scale 2^5, so
// a pair takes two accumulators per cell, 128 per lane, and two waves
// share a SIMD. Every lane reads its rows' bitplane words from global memory
// (one dword per operand and 64 individuals, coalesced along SNPs) and expands
// them in registers: no operand passes through LDS, and the waves run
// without barriers. LDS holds the phenotype's codes, which all waves share.
template <int TA, int ND, bool DUMP = false>
__device__ __forceinline__ void screen_fast_tile(const MfmaScan &S, const ScreenCut &C, const CandSink &cs, int a0,
                                                 int a1, int b0, int b1, uint32_t block0, uint32_t *wl,
                                                 float4 *mg, float2 *mg2, const ScreenDump &D = {})
{
    constexpr int NT = scr_threads<TA>(), ROW = sw_row<ND>();
    const uint32_t *sw = S.sw[ND - 1];
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, hf = lane >> 5;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int aw = a0 + SCR_A * wid;                      // the wave's first a-SNP
    const bool work = aw < a1 && (a1 < aw + SCR_A ? a1 : aw + SCR_A) - 1 > b0;
    const int Kw = S.Kp / 32, nw = S.Kl / 32;             // nw: words the loop covers (a multiple of 4)

    for (int i = tid; i < TA + 64; i += NT) {
        int sn = i < TA ? a0 + i : b0 + i - TA;
        sn = sn < S.nsnp ? sn : S.nsnp - 1;
        const ScrMarg &q = S.sm[sn];
        mg[i] = make_float4(q.n[0], q.n[1], q.s[ND - 1][0], q.s[ND - 1][1]);
        if (i < TA) mg2[i] = make_float2(q.n[2], q.s[ND - 1][2]);
    }

    v16f av[4], al[4];  // [2 bg + h]: counts, sums of v
#pragma unroll
    for (int j = 0; j < 4; j++) av[j] = al[j] = (v16f){};

    // Bitplanes through buffer descriptors (scalar base and row offset, 32-bit lane offset): one from
    // class 0 on for the A rows, whose lanes hold both classes, and class 1 for the B rows (the
    // caller checks that two planes stay below 4 GiB).
    const uint32_t row = (uint32_t)S.nsnp * 4u, plane = (uint32_t)Kw * row;  // bytes
    const uint64_t rest = 3ull * plane;
    auto rsrc = [&](uint32_t o) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(reinterpret_cast<const char *>(S.rbits) + o), 0,
                                                 (int)(rest - o < 0xFFFFFFFFull ? rest - o : 0xFFFFFFFFull), 0x00027000);
    };
    const __amdgpu_buffer_rsrc_t r0 = rsrc(0u), r1 = rsrc(plane);
    uint32_t va, vb[2];
    {
        int a = aw + (m >> 1);
        a = a < S.nsnp ? a : S.nsnp - 1;
        va = (m & 1) * plane + hf * row + (uint32_t)a * 4u;
#pragma unroll
        for (int bg = 0; bg < 2; bg++) {
            int b = b0 + 32 * bg + m;
            b = b < S.nsnp ? b : S.nsnp - 1;
            vb[bg] = hf * row + (uint32_t)b * 4u;
        }
    }
    // Software pipeline: during step t (64 individuals) the A operands and the first B operand of step
    // t + 1 are made from bits that were loaded during step t - 1, and the bits of step t + 2 are
    // requested. The requests run up to four words past the last: those lie in the padding or in the
    // plane that follows (the call-present plane after class 1), and are not used.
    struct Ops {
        v8i A, A0, A1, B0;
    };
    uint32_t xa[2], xb[2][4];
    uint32_t src = 0;  // byte offset of the step's first word within a plane
    auto load = [&](int set) {
        xa[set] = __builtin_amdgcn_raw_buffer_load_b32(r0, va, src, 0);
#pragma unroll
        for (int j = 0; j < 4; j++)
            xb[set][j] = __builtin_amdgcn_raw_buffer_load_b32(j & 1 ? r1 : r0, vb[j >> 1], src, 0);
        src += 2 * row;
    };
    auto prep = [&](int set, const uint32_t *wr, Ops &o) {
        const uint4 q0 = *reinterpret_cast<const uint4 *>(wr), q1 = *reinterpret_cast<const uint4 *>(wr + 4);
        const Fp6 t = scr_spread(xa[set] & (ND == 1 ? q1.z : wr[12])), f = scr_fill(t);
        const Fp6 f0 = {{f.d[0] & q0.x, f.d[1] & q0.y, f.d[2] & q0.z, f.d[3] & q0.w, f.d[4] & q1.x, f.d[5] & q1.y}};
        o.A = scr_op(t);
        o.A0 = scr_op(f0);
        if constexpr (ND == 2) {
            const uint4 q2 = *reinterpret_cast<const uint4 *>(wr + 8);
            const Fp6 f1 = {{f.d[0] & q1.z, f.d[1] & q1.w, f.d[2] & q2.x, f.d[3] & q2.y, f.d[4] & q2.z, f.d[5] & q2.w}};
            o.A1 = scr_op(f1);
        }
        o.B0 = scr_op(scr_spread(xb[set][0]));
    };
    auto step = [&](int set, const Ops &o) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const v8i B = j == 0 ? o.B0 : scr_op(scr_spread(xb[set][j]));
            al[j] = scr_mfma(o.A0, B, al[j]);
            av[j] = scr_mfma(o.A, B, av[j]);
            if constexpr (ND == 2) al[j] = scr_mfma32(o.A1, B, al[j]);
        }
    };
    // Masks: 0x008 MFMA, 0x002 VALU, 0x100 LDS read, 0x020 global load.
    auto fence = [&]() {
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * ND, 0);
#pragma unroll
        for (int u = 0; u < 4 + 4 * ND; u++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, ND == 1 ? 8 : 6, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    Ops o0, o1;
    if (work) {
        load(0);
        load(1);
    }
    for (int w0 = 0; w0 < nw; w0 += SCR_WIN) {
        const int wn = nw - w0 < SCR_WIN ? nw - w0 : SCR_WIN;
        if (w0) __syncthreads();
        scr_stage<NT, ROW>(wl, sw + (size_t)w0 * ROW, wn, tid);
        __syncthreads();
        if (!work) continue;
        const uint32_t *wr = wl + hf * ROW;
        prep(0, wr, o0);
        __builtin_amdgcn_sched_barrier(0);
        for (int t = 0; t < wn; t += 4, wr += 4 * ROW) {
            step(0, o0);
            prep(1, wr + 2 * ROW, o1);
            load(0);
            fence();
            step(1, o1);
            // past the window's last step: a row of the next window's place, not used
            prep(0, wr + 4 * ROW, o0);
            load(1);
            fence();
        }
    }
    if (!work) return;

    // Lane: pairs a = aw + 4j + 2hf + p, b = b0 + 32 bg + m; [2bg + h][4j + 2p + g] = X[g][h].
    uint32_t bits = 0;
    const float4 mb[2] = {mg[TA + m], mg[TA + 32 + m]};
    static_for<16>([&](auto k) {
        constexpr int K = decltype(k)::value, j = K / 4, p = K / 2 % 2, bg = K % 2, e = 4 * j + 2 * p;
        const int ia = SCR_A * wid + 4 * j + 2 * hf + p;
        const float4 ma = mg[ia];
        const float2 ma2 = mg2[ia];
        float n[9], s[9];
        auto fill = [&](float c[9], const v16f &x0, const v16f &x1, float a_0, float a_1, float a_2, float b_0, float b_1) {
            c[0] = x0[e];
            c[1] = x1[e];
            c[3] = x0[e + 1];
            c[4] = x1[e + 1];
            c[2] = a_0 - c[0] - c[1];
            c[5] = a_1 - c[3] - c[4];
            c[6] = b_0 - c[0] - c[3];
            c[7] = b_1 - c[1] - c[4];
            c[8] = a_2 - c[6] - c[7];
        };
        fill(n, av[2 * bg], av[2 * bg + 1], ma.x, ma.y, ma2.x, mb[bg].x, mb[bg].y);
        fill(s, al[2 * bg], al[2 * bg + 1], ma.z, ma.w, ma2.y, mb[bg].z, mb[bg].w);
        if constexpr (DUMP) {
            const int a = aw + 4 * j + 2 * hf + p, b = b0 + 32 * bg + m;
            if (a < a1 && b < b1 && a > b) screen_dump(D, S, a, b, n, s);
            return;
        }
        float u = 0.0f;
#pragma unroll
        for (int c = 0; c < 9; c++) u = __builtin_fmaf(s[c] * s[c], rcp_above(n[c]), u);
        const float thr = __builtin_fmaf(C.slope2, scr_nfac2(n), C.thr0);
        bool keep = !(u <= thr);
        if (__ballot(keep) != 0ull) {
            const int a = aw + 4 * j + 2 * hf + p, b = b0 + 32 * bg + m;
            keep = keep & (a < a1) & (b < b1) & (a > b);
            keep = keep && screen_bound(n, s, C.nv, C.sst, C);
            bits |= keep ? 1u << K : 0u;
        }
        __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (DUMP) return;
    scr_append<16>(cs, bits, block0, wid, S.tag, [&](int k, int &a, int &b) {
        a = aw + 4 * (k >> 2) + 2 * hf + (k >> 1 & 1);
        b = b0 + 32 * (k & 1) + m;
    });
}

template <int TA, int ND>
__global__ __launch_bounds__(scr_threads<TA>(), 2) void screen_fast_kernel(const ScreenArgs A)
{
    __shared__ __attribute__((aligned(16))) uint32_t wl[SCR_LDS_ROWS * sw_row<ND>()];
    __shared__ float4 mg[TA + 64];
    __shared__ float2 mg2[TA];
    const int t = xcd_tile(blockIdx.x, A.ntiles);
    const int4 T = A.tiles[t];
    screen_fast_tile<TA, ND>(A.S, A.cut, A.cs, T.x, T.y, T.z, T.w, (uint32_t)(A.tile0 + t) * scr_blocks(TA, 64, false),
                             wl, mg, mg2);
}

// ------------------------------------------------------------- GENERAL ----
// Tile TA a x 32 b with missing calls (a SPARSE tile, whose SNPs miss few calls, is two of them). Each
// wave owns 16 a x 32 b and contracts three masks of both sides with the count and the two
// digits: 27 v_mfma_f32_16x16x128_f8f6f4 per 16 x 16 pairs and 128 individuals (the exact tile: 40 INT8
// MACs per pair and individual, here 27 at twice the rate). The 16 x 16 shape puts a pair's 18 accumulators
// into one lane whatever the number of rows per a-SNP: row m of A is a-SNP m, one
// block per class and weight; lane l holds column l % 16 and rows 4 (l / 16) + i. 144 accumulators.
// The masks are the two rarest classes and, with NC, the missing calls (the commonest class's cells follow from
// those and the SNPs' own sums: 36 more instructions a pair slot), otherwise the commonest class itself. Missing calls
// are the sparser operand, and the matrix cores' power bounds the clock: from N = 3000 the scan gains (kernel time of
// NC over not, 1 % missing calls: N = 500 1.09, 2000 1.03, 3000 0.99, 4000 0.97, 8000 0.95, 20000 0.92).
// SST of a pair's complete cases is at least Z_a + Z_b - Z_all (Z the sums of q^2 over an
// SNP's calls), less the mean's part, T^2 / N with T the sum of q: |T| / sqrt N <= delta |sum v| / sqrt N + eps.
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f scr_mfma16(const v8i &a, const v8i &b, const v4f &c)
{
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 2, 2, 0, 0, 0, 0);
}
__device__ __forceinline__ v4f scr_mfma16x32(const v8i &a, const v8i &b, const v4f &c)
{
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 2, 2, 0, 0x84848484, 0, 0x7f7f7f7f);
}

template <int TA, int ND, bool NC, bool DUMP = false>
__device__ __forceinline__ void screen_gen_tile(const MfmaScan &S, const ScreenCut &C, const CandSink &cs, int a0, int a1,
                                                int b0, int b1, uint32_t block0, uint32_t *wl, float4 *mg,
                                                const ScreenDump &D = {})
{
    constexpr int TB = 32, NT = scr_threads<TA>(), ROW = sw_row<ND>();
    const uint32_t *sw = S.sw[ND - 1];
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, kq = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int al = SCR_A * wid, aw = a0 + al, bw = b0;
    const bool work = aw < a1 && (a1 < aw + SCR_A ? a1 : aw + SCR_A) - 1 > bw;
    const int Kw = S.Kp / 32, nw = S.Kl / 32;

    float *mz = reinterpret_cast<float *>(mg);  // without NC: the sums of z alone
    for (int i = tid; i < TA + TB; i += NT) {
        int sn = i < TA ? a0 + i : b0 + i - TA;
        sn = sn < S.nsnp ? sn : S.nsnp - 1;
        const ScrMarg &q = S.sm[sn];
        if constexpr (!NC) {
            mz[i] = q.zs;
            continue;
        }
        const float *qs = q.s[ND - 1];
        mg[i] = make_float4(q.n[0], q.n[1], qs[0], qs[1]);
        // a: the commonest class; b: missing calls
        mg[TA + TB + i] = i < TA ? make_float4(q.n[2], qs[2], q.zs, 0.0f)
                                 : make_float4(C.N - q.n[0] - q.n[1] - q.n[2], C.vs - qs[0] - qs[1] - qs[2], q.zs, 0.0f);
    }

    v4f av[2][9], as[2][9];  // [b group][3 g + h]: counts, sums of v
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 9; j++) av[i][j] = as[i][j] = (v4f){};

    // bitplanes through one buffer descriptor per class (scalar base and row offset, 32-bit lane offset)
    const uint32_t row = (uint32_t)S.nsnp * 4u, plane = (uint32_t)Kw * row;  // bytes
    auto rsrc = [&](int g) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(reinterpret_cast<const char *>(S.rbits) + (size_t)g * plane), 0,
                                                 (int)plane, 0x00027000);
    };
    const __amdgpu_buffer_rsrc_t r[3] = {rsrc(0), rsrc(1), rsrc(2)};
    uint32_t va, vb[2];
    {
        const int a = aw + m < S.nsnp ? aw + m : S.nsnp - 1;
        va = kq * row + (uint32_t)a * 4u;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int b = bw + 16 * i + m < S.nsnp ? bw + 16 * i + m : S.nsnp - 1;
            vb[i] = kq * row + (uint32_t)b * 4u;
        }
    }
    // Software pipeline over steps of 128 individuals, in three phases, one per class g of the a-SNPs, of three
    // groups of six MFMAs (one per B operand): the low digit, the count, the high digit. A group's
    // operand is made one or two groups before it and dies with it, so that at most four A operands are
    // live beside the six of B; the last group of a step makes the next step's B operands
    // in the registers of this one's.
    struct Weights {
        uint4 q0, q1, q2;
        uint32_t v;
    };
    uint32_t xa[3], xb[6];
    v8i B[6];
    uint32_t src = 0;
    const uint32_t last = (uint32_t)(nw - 4) * row;
    auto loadB = [&]() {
#pragma unroll
        for (int j = 0; j < 6; j++) xb[j] = __builtin_amdgcn_raw_buffer_load_b32(r[j >> 1], vb[j & 1], src, 0);
    };
    auto loadA = [&](int g) { xa[g] = __builtin_amdgcn_raw_buffer_load_b32(r[g], va, src, 0); };
    // the word of B operand j = 2 h + b group; h = 2: no call, or the commonest class (the rest of the called)
    auto word = [&](int j) { return j < 4 ? xb[j] : NC ? ~xb[j] : xb[j] & ~xb[j - 4] & ~xb[j - 2]; };
    auto low = [&](const Fp6 &f, const Weights &w) {
        return scr_op({{f.d[0] & w.q0.x, f.d[1] & w.q0.y, f.d[2] & w.q0.z, f.d[3] & w.q0.w, f.d[4] & w.q1.x,
                        f.d[5] & w.q1.y}});
    };
    auto high = [&](const Fp6 &f, const Weights &w) {
        return scr_op({{f.d[0] & w.q1.z, f.d[1] & w.q1.w, f.d[2] & w.q2.x, f.d[3] & w.q2.y, f.d[4] & w.q2.z,
                        f.d[5] & w.q2.w}});
    };
    if (work) {
        loadA(0);
        loadB();
    }
    for (int w0 = 0; w0 < nw; w0 += SCR_WIN) {
        const int wn = nw - w0 < SCR_WIN ? nw - w0 : SCR_WIN;
        if (w0) __syncthreads();
        scr_stage<NT, ROW>(wl, sw + (size_t)w0 * ROW, wn, tid);
        __syncthreads();
        if (!work) continue;
        const uint32_t *wr = wl + kq * ROW;
        Weights w;
        auto weights = [&](int part) {
            if (part == 0) {
                w.v = wr[6 * ND];
                w.q0 = *reinterpret_cast<const uint4 *>(wr);
                w.q1.x = wr[4];
                w.q1.y = wr[5];
            } else if (ND == 2) {
                w.q1.z = wr[6];
                w.q1.w = wr[7];
                w.q2 = *reinterpret_cast<const uint4 *>(wr + 8);
            }
        };
        weights(0);
        weights(1);
        Fp6 t = scr_spread(xa[0] & w.v), f = scr_fill(t);
        v8i A0 = low(f, w);
#pragma unroll
        for (int j = 0; j < 6; j++) B[j] = scr_op(scr_spread(word(j)));
        loadA(1);
        loadA(2);
        __builtin_amdgcn_sched_barrier(0);
        // Masks: 0x008 MFMA, 0x002 VALU.
        auto fence = [&](auto nv) {
#pragma unroll
            for (int u = 0; u < 6; u++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, decltype(nv)::value, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        using std::integral_constant;
        for (int wi = 0; wi < wn; wi += 4) {
            uint32_t a01 = 0;
            static_for<3>([&](auto gg) {
                constexpr int g = decltype(gg)::value, gn = (g + 1) % 3;
                if (g == 0) {  // request the next step's words
                    a01 = xa[0] | xa[1];
                    src = src + 4 * row < last ? src + 4 * row : last;
                    loadA(0);
                    loadB();
                }
                if (g == 2) {
                    wr += 4 * ROW;  // past the window's last step: not used
                    weights(0);
                }
#pragma unroll
                for (int j = 0; j < 6; j++) as[j & 1][3 * g + (j >> 1)] = scr_mfma16(A0, B[j], as[j & 1][3 * g + (j >> 1)]);
                const Fp6 tn = scr_spread(gn < 2 ? xa[gn] & w.v : NC ? ~xa[2] & w.v : xa[2] & ~a01 & w.v);
                if (g == 2) {
                    loadA(1);
                    loadA(2);
                }
                fence(integral_constant<int, 2>{});
                if constexpr (ND == 1) A0 = low(scr_fill(tn), w);
#pragma unroll
                for (int j = 0; j < 6; j++) {
                    av[j & 1][3 * g + (j >> 1)] = scr_mfma16(scr_op(t), B[j], av[j & 1][3 * g + (j >> 1)]);
                    if (ND == 1 && g == 2) {
                        B[j] = scr_op(scr_spread(word(j)));
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                if (ND == 1 && g < 2) fence(integral_constant<int, 3>{});
                if constexpr (ND == 2) {
                    const v8i A1 = high(f, w);
                    if (g == 2) weights(1);
                    const Fp6 fn = scr_fill(tn);
                    fence(integral_constant<int, 3>{});
                    A0 = low(fn, w);
#pragma unroll
                    for (int j = 0; j < 6; j++) {
                        as[j & 1][3 * g + (j >> 1)] = scr_mfma16x32(A1, B[j], as[j & 1][3 * g + (j >> 1)]);
                        if (g == 2) {
                            B[j] = scr_op(scr_spread(word(j)));
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                    f = fn;
                    if (g < 2) fence(integral_constant<int, 1>{});
                }
                t = tn;
            });
        }
    }
    if (!work) return;

    // Lane: pairs a = aw + 4 kq + i, b = bw + 16 bg + m.
    uint32_t bits = 0;
    float4 mb[2] = {}, mb2[2] = {};
#pragma unroll
    for (int j = 0; j < 2; j++) {
        if (NC) mb[j] = mg[TA + 16 * j + m], mb2[j] = mg[TA + TB + TA + 16 * j + m];
        else mb2[j].z = mz[TA + 16 * j + m];
    }
    static_for<8>([&](auto k) {
        constexpr int K = decltype(k)::value, i = K / 2, bg = K % 2;
        const int ia = al + 4 * kq + i;
        float4 ma = {}, ma2 = {};
        if (NC) ma = mg[ia], ma2 = mg[TA + TB + ia];
        else ma2.z = mz[ia];
        float n[9], s[9];
        // the table from the sums over {0, 1, no call}^2 and the SNPs' own; returns its total
        auto fill = [&](float c[9], const v4f (&X)[9], float a_0, float a_1, float a_2, float b_0, float b_1, float b_m) {
            c[0] = X[0][i];
            c[1] = X[1][i];
            c[3] = X[3][i];
            c[4] = X[4][i];
            c[2] = a_0 - c[0] - c[1] - X[2][i];
            c[5] = a_1 - c[3] - c[4] - X[5][i];
            c[6] = b_0 - c[0] - c[3] - X[6][i];
            c[7] = b_1 - c[1] - c[4] - X[7][i];
            const float lost = b_m - X[8][i];  // called in a, not in b
            c[8] = a_2 - c[6] - c[7] - (lost - X[2][i] - X[5][i]);
            return a_0 + a_1 + a_2 - lost;
        };
        float nc = 0.0f, tc = 0.0f;
        if constexpr (NC) {
            nc = fill(n, av[bg], ma.x, ma.y, ma2.x, mb[bg].x, mb[bg].y, mb2[bg].x);
            tc = fill(s, as[bg], ma.z, ma.w, ma2.y, mb[bg].z, mb[bg].w, mb2[bg].y);
        } else {
#pragma unroll
            for (int c = 0; c < 9; c++) {
                n[c] = av[bg][c][i];
                s[c] = as[bg][c][i];
                nc += n[c];
                tc += s[c];
            }
        }
        if constexpr (DUMP) {
            const int a = aw + 4 * kq + i, b = bw + 16 * bg + m;
            if (a < a1 && b < b1 && a > b) screen_dump(D, S, a, b, n, s);
            return;
        }
        tc = __builtin_fmaf(C.c0, nc, tc);
        const float zlow = ma2.z + mb2[bg].z - C.zall;
        float u = 0.0f;
#pragma unroll
        for (int c = 0; c < 9; c++) u = __builtin_fmaf(s[c] * s[c], rcp_above(n[c]), u);
        // SST from below: (x + eps)^2 <= 2 x^2 + 2 eps^2
        const float sst0 = zlow * C.zunit - 2.0f * (tc * tc * rcp_above(nc) + C.eps * C.eps);
        const float kap = __builtin_fmaf(C.kslope2, scr_nfac2(n), C.kap0);
        bool keep = !((u <= kap * sst0 - C.kroot) & (2.0f * nc >= C.N));
        if (__ballot(keep) != 0ull) {
            const int a = aw + 4 * kq + i, b = bw + 16 * bg + m;
            keep = keep & (a < a1) & (b < b1) & (a > b);
            const float rt = fabsf(tc) * __builtin_amdgcn_rsqf(nc) * 1.0001f + C.eps;
            keep = keep && screen_bound(n, s, 64.0f * nc, zlow * C.zunit - rt * rt, C);
            bits |= keep ? 1u << K : 0u;
        }
        __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (DUMP) return;
    scr_append<8>(cs, bits, block0, wid, S.tag, [&](int k, int &a, int &b) {
        a = aw + 4 * kq + (k >> 1);
        b = bw + 16 * (k & 1) + m;
    });
}

// Whether a scan of Kl individuals (a multiple of 128) contracts the missing calls. Only with 64-row tiles.
__host__ __device__ constexpr bool scr_nocall(int Kl) { return Kl >= 3000; }

// The workgroup's half of 32 b (or the whole) of a tile: b range and first block. False: no b-SNPs.
template <int TA>
__device__ __forceinline__ bool scr_half(int h, int halves, uint32_t tile, int &b0, int &b1, uint32_t &block0)
{
    b0 += 32 * h;
    block0 = (tile * halves + h) * (TA / 32);
    const bool any = b0 < b1;
    b1 = b1 < b0 + 32 ? b1 : b0 + 32;
    return any;
}

template <int TA, int ND, bool NC>
__global__ __launch_bounds__(scr_threads<TA>(), 2) void screen_gen_kernel(const ScreenArgs A)
{
    __shared__ __attribute__((aligned(16))) uint32_t wl[SCR_GEN_ROWS * sw_row<ND>()];
    __shared__ float4 mg[2 * (TA + 32)];
    const int t = xcd_tile(blockIdx.x, A.ntiles * A.halves);
    int4 T = A.tiles[t / A.halves];
    uint32_t block0;
    if (!scr_half<TA>(t % A.halves, A.halves, (uint32_t)(A.tile0 + t / A.halves), T.z, T.w, block0)) return;
    screen_gen_tile<TA, ND, NC>(A.S, A.cut, A.cs, T.x, T.y, T.z, T.w, block0, wl, mg);
}

// The tiles above without decisions.
template <int TA, int ND>
__global__ __launch_bounds__(scr_threads<TA>(), 2) void screen_fast_dump(const ScreenArgs A, const ScreenDump D)
{
    __shared__ __attribute__((aligned(16))) uint32_t wl[SCR_LDS_ROWS * sw_row<ND>()];
    __shared__ float4 mg[TA + 64];
    __shared__ float2 mg2[TA];
    const int4 T = A.tiles[blockIdx.x];
    screen_fast_tile<TA, ND, true>(A.S, A.cut, A.cs, T.x, T.y, T.z, T.w, 0, wl, mg, mg2, D);
}

template <int TA, int ND, bool NC>
__global__ __launch_bounds__(scr_threads<TA>(), 2) void screen_gen_dump(const ScreenArgs A, const ScreenDump D)
{
    __shared__ __attribute__((aligned(16))) uint32_t wl[SCR_GEN_ROWS * sw_row<ND>()];
    __shared__ float4 mg[2 * (TA + 32)];
    const int4 T = A.tiles[blockIdx.x];
    screen_gen_tile<TA, ND, NC, true>(A.S, A.cut, A.cs, T.x, T.y, T.z, T.w, 0, wl, mg, D);
}

// After the candidates of a launch are resolved: the list is emptied for the next one.
__global__ void empty_list(uint32_t *count, uint32_t cap, unsigned long long *total)
{
    *total += *count < cap ? *count : cap;
    *count = 0u;
}

// --------------------------------------------------------------- redo ----
// Blocks that the screen handed back, through the exact tiles of 32 rows (16, where only one of the two waves asked for
// it): a workgroup per block where the host knows their number (single scans), otherwise a persistent grid. (One exact
// tile per wave, half of its rows unused, N = 3000, M = 30000 with 1.5 % of the pairs hits: 44.3 ms; a persistent grid over
// blocks 33.3, now 32.6.) Each marked block is in the list once; its mask is left at 0 for the next scan.
struct RedoArgs {
    MfmaScan S;               // single scans
    const MfmaScan *scans;    // batches: by scan id
    HitSink hs;
    const int4 *tiles;        // single scans {a0, a1, b0, b1}; batches {a0, b0, extents, scan}
    const uint32_t *count;
    const uint32_t *redo;
    uint32_t *mask;
};

template <int TA, int TB, bool GEN, bool BATCH>
__global__ __launch_bounds__(256, 2) void redo_kernel(const RedoArgs A)
{
    static_assert(fast_threads<32>() == 256 && general_threads<32>() == 256, "threads of the 32-row tiles");
    constexpr int RB = GEN ? 32 : 64, NBA = TA / 32, NBLK = scr_blocks(TA, TB, GEN);
    __shared__ __attribute__((aligned(16))) uint8_t lds[GEN ? general_lds<32>() : fast_lds<32>()];
    const uint32_t n = A.count[1];
    const DumpSink nodump = {};
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
        const uint32_t r = __builtin_amdgcn_readfirstlane(A.redo[gridDim.x == n ? xcd_tile(i, n) : i]), half = __builtin_amdgcn_readfirstlane(A.mask[r]);
        __syncthreads();  // the mask is read, and the previous tile is done with LDS
        if (threadIdx.x == 0) A.mask[r] = 0u;
        int4 T = A.tiles[r / NBLK];
        HitSink hs = A.hs;
        int sc = 0;
        if (BATCH) {
            sc = __builtin_amdgcn_readfirstlane(T.w);
            T = make_int4(T.x, T.x + (T.z & 255), T.y, T.y + ((T.z >> 8) & 255));
        }
        const MfmaScan &S = BATCH ? A.scans[sc] : A.S;
        hs.tag = S.tag;
        const int k = (int)(r % NBLK);
        int a0 = __builtin_amdgcn_readfirstlane(T.x) + 32 * (k % NBA), a1 = __builtin_amdgcn_readfirstlane(T.y);
        int b0 = __builtin_amdgcn_readfirstlane(T.z) + RB * (k / NBA), b1 = __builtin_amdgcn_readfirstlane(T.w);
        const int end = a0 + (half & 2u ? 32 : SCR_A);
        a0 += half & 1u ? 0 : SCR_A;
        a1 = a1 < end ? a1 : end;
        b1 = b1 < b0 + RB ? b1 : b0 + RB;
        if (a0 >= a1 || b0 >= b1 || a1 - 1 <= b0) continue;
        if constexpr (GEN)
            mfma_general_tile<32, false>(S, hs, nodump, a0, a1, b0, b1, lds);
        else
            mfma_fast_tile<32, false>(S, hs, nodump, a0, a1, b0, b1, lds);
    }
}

// --------------------------------------------------------------- resolve ----
// The candidates' exact tables, one wave (or a part of it) per candidate: its
// lanes take the bitplane words of both SNPs in turn and sum V (the counts),
// the three limbs of q (and the four of z for pairs with missing calls) with
// 4 x 8-bit dot products, exactly as the tiles' MFMAs do, in INT32. The lanes'
// sums are added up, and lane i keeps candidate i of the wave's run, so that
// the FP64 decision runs once for all of them, on up to 64 lanes.
struct ResolveArgs {
    MfmaScan S;               // single scans
    const MfmaScan *scans;    // batches: by scan id
    HitSink hs;
    const int4 *cand;
    const uint32_t *count;
    uint32_t cap;
    int group;                // lanes per candidate
};

// Sums of t over groups of G lanes, in all of them: within 16 lanes each addition takes its other operand from another
// lane (DPP), beyond through LDS. Step by step for all values together, so that they hide each other's latency.
// (Values one after the other, up to six dependent rounds through LDS each: 4,000 candidates with missing calls at N = 1237
// 46 -> 21 us; 3,000 without at N = 500 18.5 -> 15.5 us, most of that the chain of loads and the FP64 statistics.)
template <int NV>
__device__ __forceinline__ void resolve_sum(int (&t)[NV], int G)
{
    auto add = [&](auto ctrl) {
#pragma unroll
        for (int i = 0; i < NV; i++) t[i] += __builtin_amdgcn_mov_dpp(t[i], decltype(ctrl)::value, 0xF, 0xF, true);
    };
    using std::integral_constant;
    add(integral_constant<int, 0xB1>{});                 // lane ^ 1
    add(integral_constant<int, 0x4E>{});                 // lane ^ 2
    if (G >= 8) add(integral_constant<int, 0x141>{});    // the other half of 8 lanes, mirrored
    if (G >= 16) add(integral_constant<int, 0x140>{});   // the other half of 16 lanes, mirrored
    for (int o = 16; o < G; o *= 2) {
        int v[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) v[i] = __shfl_xor(t[i], o);
#pragma unroll
        for (int i = 0; i < NV; i++) t[i] += v[i];
    }
}

// GEN: pairs of tiles with missing calls (the classes 0, 1, NM of both SNPs and
// the sum of z); otherwise classes 0 and 1 and the SNPs' marginals. G lanes
// share a candidate (a power of two, 64 from 33 words on), so that a wave
// takes 64 / G candidates of a small cohort at a time.
template <bool GEN, bool BATCH>
__global__ __launch_bounds__(256) void resolve_kernel(const ResolveArgs A)
{
    constexpr int NG = GEN ? 3 : 2, NX = NG * NG, NZ = GEN ? 4 : 0, NV = 4 * NX + NZ;
    const uint32_t n = A.count[0] < A.cap ? A.count[0] : A.cap;
    const uint32_t nwave = gridDim.x * 4u, wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, G = A.group, sub = lane / G, gl = lane % G, step = 64 / G;
    uint32_t per = (n + nwave - 1) / nwave;
    per = (per + step - 1) / step * step;
    per = per < 64u ? per : 64u;
    for (uint32_t c0 = wave * per; c0 < n; c0 += nwave * per) {
        const int m = (int)(n - c0 < per ? n - c0 : per);
        int keep[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) keep[i] = 0;
        const int4 mine = A.cand[c0 + (lane < m ? lane : 0)];
        for (int u = 0; u < m; u += step) {
            const int c = u + sub;
            const int a = __shfl(mine.x, c), b = __shfl(mine.y, c);
            const MfmaScan &S = BATCH ? A.scans[__shfl(mine.z, c)] : A.S;
            const bool on = c < m && a != b;
            const int Kw = S.Kp / 32, nw = on ? S.Kl / 32 : 0;
            // bits by SNP, or the bitplanes where memory was short
            const bool by = S.sbits != nullptr;
            const uint32_t *bits = by ? S.sbits : S.bits;
            const size_t plane = (size_t)Kw * S.nsnp, sw = by ? 1 : S.nsnp, oa = (size_t)a * (by ? Kw : 1), ob = (size_t)b * (by ? Kw : 1);
            int t[NV];
#pragma unroll
            for (int i = 0; i < NV; i++) t[i] = 0;
            for (int w = gl; w < nw; w += G) {
                uint32_t x[NX];
                {
                    uint32_t ga[NG], hb[NG];
#pragma unroll
                    for (int g = 0; g < NG; g++) {
                        ga[g] = bits[g * plane + oa + w * sw];
                        hb[g] = bits[g * plane + ob + w * sw];
                    }
#pragma unroll
                    for (int g = 0; g < NG; g++)
#pragma unroll
                        for (int h = 0; h < NG; h++) x[g * NG + h] = ga[g] & hb[h];
                }
                const int8_t *wp = S.wts + 32 * w;
#pragma unroll
                for (int hh = 0; hh < 2; hh++) {
                    int4 l[4], z[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        l[i] = *reinterpret_cast<const int4 *>(wp + (size_t)i * S.Kp + 16 * hh);
                        if (GEN) z[i] = *reinterpret_cast<const int4 *>(wp + (size_t)(4 + i) * S.Kp + 16 * hh);
                    }
#pragma unroll
                    for (int i = 0; i < NX; i++) {
                        const v4i e = expand16<false>((x[i] >> (16 * hh)) & 0xFFFFu);
#pragma unroll
                        for (int q = 0; q < 4; q++) {
#pragma unroll
                            for (int k = 0; k < 4; k++) {
                                const int lw = k == 0 ? l[q].x : k == 1 ? l[q].y : k == 2 ? l[q].z : l[q].w;
                                t[4 * i + q] = __builtin_amdgcn_sdot4(e[k], lw, t[4 * i + q], false);
                            }
                        }
                        if (GEN && i == NX - 1) {
#pragma unroll
                            for (int q = 0; q < 4; q++)
#pragma unroll
                                for (int k = 0; k < 4; k++) {
                                    const int zw = k == 0 ? z[q].x : k == 1 ? z[q].y : k == 2 ? z[q].z : z[q].w;
                                    t[4 * NX + q] = __builtin_amdgcn_sdot4(e[k], zw, t[4 * NX + q], false);
                                }
                        }
                    }
                }
            }
            resolve_sum<NV>(t, G);
#pragma unroll
            for (int i = 0; i < NV; i++) {
                const int v = G < 64 ? __shfl(t[i], (lane - u) * G) : t[i];
                keep[i] = lane >= u && lane < u + step ? v : keep[i];
            }
        }
        const bool valid = lane < m && mine.x != mine.y;
        bool hit = false;
        DevHit h;
        HitSink hs = A.hs;
        if (valid) {
            const MfmaScan &S = BATCH ? A.scans[mine.z] : A.S;
            hs.tag = S.tag;
            int xc[3][3], nc[9];
            double xs[3][3], sd[9], sq;
#pragma unroll
            for (int g = 0; g < NG; g++)
#pragma unroll
                for (int k = 0; k < NG; k++) {
                    const int *v = keep + 4 * (g * NG + k);
                    xc[g][k] = v[0];
                    xs[g][k] = (double)v[1] + 256.0 * (double)v[2] + 65536.0 * (double)v[3];
                }
            if (GEN) {
                const int *z = keep + 4 * NX;
                sq = ((double)z[0] + 256.0 * (double)z[1] + 65536.0 * (double)z[2] + 16777216.0 * (double)z[3]) * S.zunit;
            } else {
                const Marg &ma = S.marg[mine.x], &mb = S.marg[mine.y];
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    xc[g][2] = ma.n[g];
                    xc[2][g] = mb.n[g];
                    xs[g][2] = (double)ma.q[g];
                    xs[2][g] = (double)mb.q[g];
                }
                xc[2][2] = S.nV;
                xs[2][2] = S.qVd;
                sq = S.sqV;
            }
            cells_from_x(xc, nc);
            cells_from_x(xs, sd);
            hit = confirm64(hs, mine.x, mine.y, nc, sd, sq, h);
        }
        append_hit(hs, hit, h);
    }
}

}  // namespace epi
