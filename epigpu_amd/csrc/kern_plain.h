// Plain popcount form of the pair scan (gfx950 VALU).
//
// Genotypes are class bitplanes (bit k of word w = individual 32w + k) laid
// out [plane][word][snp]. A workgroup of NT threads takes a tile of NT/16 x 64
// pairs, every thread 2 x 2 of them, and goes through the individuals a word
// (32) at a time: it writes y_k [k in B_h] of its 64 b-SNPs to LDS (two
// buffers, one barrier per word) and holds its a-SNPs' words in registers.
//   counts  X[g][h] += popcount(A_g & V & B_h)      (AND + v_bcnt per word)
//   sums    X[g][h] += [k in A_g] * (y_k [k in B_h])         (masked FP32 FMA)
// FP32 partial sums are promoted to FP64 after every word. The two bitplanes
// of a SNP hold its two rarest genotype classes and the most common class is
// derived (by subtraction from the NM totals), so a small cell never inherits
// the rounding error of a large one. FAST tiles use the planes {0,1}; GENERAL
// tiles add the NM plane and the sum of y^2 over complete cases. The per-pair
// epilogue is shared with the MFMA form.
//
// What bounds it: VALU issue, at half the rate for instructions with a scalar
// operand, shifts left, bit-field extracts, conversions and popcounts (two waves
// of a SIMD issue FMAs, adds, ANDs and shifts right together where all operands
// are vector registers or literals: 0.37-0.39 a cycle measured in registers,
// 0.24 with a scalar factor). So the factor [k in A_g] of an FMA is one AND: bit
// 16 + j of an a-word, kept in its place, is as FP32 the (denormal) number
// 2^(j - 133), and yw holds y_k 2^(126 - j) for j = k mod 8. Both factors are
// powers of two away from [bit] and y_k, so every partial sum is the plain one
// times PLAIN_SCALE, with the same roundings. 2 x 2 pairs a thread leave FAST
// tiles four waves per SIMD (128 registers); 4 x 2 with two waves took 5-10 % more.
// N = 4000, M = 8000: 17.3 ms with every mask extracted and converted by each
// thread, 12.6 ms; N = 1500, M = 6000: 3.8 -> 3.0 ms; N = 1500, M = 4001, 2 %
// missing calls: 4.3 -> 3.3 ms. At that rate the FMAs alone are 0.68 of the first.
#pragma once

#include "epilogue.h"
#include "kern_mfma.h"  // Marg, xcd_tile

namespace epi {

constexpr double PLAIN_SCALE = 1.0 / 128;  // of the partial sums (2^(126 - j + 16 + j - 149))

// A factor y of individual k (|y| < 1) as the kernel reads it.
inline float plain_weight(float y, int k) { return y * (0x1p126f / (float)(1 << (k & 7))); }

// Factors of N individuals of a word, the same for a whole wave, through the scalar cache.
template <int N>
using plain_y = float __attribute__((ext_vector_type(N), aligned(4)));
template <int N>
__device__ __forceinline__ plain_y<N> plain_sload(const float *p)
{
    return *reinterpret_cast<const __attribute__((address_space(4))) plain_y<N> *>(reinterpret_cast<uintptr_t>(p));
}

// LDS of a tile: y_k [k in B_h] (and y_k^2 [k in NM] of GENERAL tiles) of 32 individuals and 64 SNPs, twice.
template <bool FAST>
struct PlainLds {
    typedef float row __attribute__((ext_vector_type(FAST ? 2 : 4)));
    __attribute__((aligned(16))) row y[2][32][64];
};

struct PlainScan {          // one dataset x one phenotype
    const uint32_t *bits;   // [3][Kw][nsnp]
    const float *yw;        // [2][Kp] centred FP32 phenotype y (0 where missing) and y^2, as plain_weight
    const uint32_t *vbits;  // [Kw] phenotype-present bits
    const Marg *marg;       // [nsnp]
    int nsnp;
    int Kw;
    int nw;                 // words that hold individuals
    int nV;
    int tag;                // written into the hits
    double ysV;             // sum of yc over present
    double y2V;             // sum of yc^2 over present
};

struct PlainArgs {
    PlainScan S;
    const int4 *tiles;
    int ntiles;
    HitSink hs;
    DumpSink ds;
};

template <int NT, bool FAST, bool DUMP>
__device__ __forceinline__ void plain_tile(const PlainScan &P, const HitSink &hs, const DumpSink &dsk, int a0, int a1,
                                           int b0, int b1, PlainLds<FAST> &lds)
{
    constexpr int NP = FAST ? 2 : 3, PA = 2, PB = 2, NI = 2048 / NT;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int nsnp = P.nsnp;
    const size_t plane = (size_t)P.Kw * nsnp;
    // staging: lane = b-SNP, a wave takes eight individuals of the word
    const int sl = threadIdx.x & 63, sk = NI * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t sb = b0 + sl < nsnp ? b0 + sl : nsnp - 1;
    uint32_t as[PA], bs[PB];
#pragma unroll
    for (int i = 0; i < PA; i++) as[i] = a0 + PA * ty + i < nsnp ? a0 + PA * ty + i : nsnp - 1;
#pragma unroll
    for (int j = 0; j < PB; j++) bs[j] = b0 + PB * tx + j < nsnp ? b0 + PB * tx + j : nsnp - 1;

    int cnt[PA][PB][NP][NP];
    float sf[PA][PB][NP][NP];
    double sd[PA][PB][NP][NP];
    float qf[PA][PB];
    double qd[PA][PB];
#pragma unroll
    for (int i = 0; i < PA; i++)
#pragma unroll
        for (int j = 0; j < PB; j++) {
            qf[i][j] = 0.0f;
            qd[i][j] = 0.0;
#pragma unroll
            for (int g = 0; g < NP; g++)
#pragma unroll
                for (int h = 0; h < NP; h++) {
                    cnt[i][j][g][h] = 0;
                    sf[i][j][g][h] = 0.0f;
                    sd[i][j][g][h] = 0.0;
                }
        }

    uint32_t sw[NP];  // the staged b-SNP's words
    auto load = [&](int w) {
        const uint32_t *row = P.bits + (size_t)w * nsnp;
#pragma unroll
        for (int h = 0; h < NP; h++) sw[h] = (row + h * plane)[sb];
    };
    auto stage = [&](int w) {
        const auto y8 = plain_sload<NI>(P.yw + 32 * w + sk);
        plain_y<NI> q8 = {};
        if (!FAST) q8 = plain_sload<NI>(P.yw + 32 * (P.Kw + w) + sk);
#pragma unroll
        for (int k = 0; k < NI; k++) {
            typename PlainLds<FAST>::row r;
#pragma unroll
            for (int h = 0; h < NP; h++) {
                const int m = __builtin_amdgcn_sbfe((int)(sw[h] >> sk), k, 1);
                r[h] = __int_as_float(m & __float_as_int(y8[k]));
                if (h == 2) r[NP] = __int_as_float(m & __float_as_int(q8[k]));
            }
            lds.y[w & 1][sk + k][sl] = r;
        }
    };
    uint32_t aw[PA][NP], bw[PB][NP], v;
    auto words = [&](int w) {
        const uint32_t *row = P.bits + (size_t)w * nsnp;
        v = P.vbits[w];
#pragma unroll
        for (int g = 0; g < NP; g++) {
#pragma unroll
            for (int i = 0; i < PA; i++) aw[i][g] = (row + g * plane)[as[i]];
#pragma unroll
            for (int j = 0; j < PB; j++) bw[j][g] = (row + g * plane)[bs[j]];
        }
    };

    load(0);
    __syncthreads();  // an earlier tile is done with LDS
    stage(0);
    if (P.nw > 1) load(1);
    words(0);
    __syncthreads();
    for (int w = 0; w < P.nw; w++) {
        if (w + 1 < P.nw) stage(w + 1);
        if (w + 2 < P.nw) load(w + 2);
#pragma unroll
        for (int i = 0; i < PA; i++)
#pragma unroll
            for (int j = 0; j < PB; j++)
#pragma unroll
                for (int g = 0; g < NP; g++)
#pragma unroll
                    for (int h = 0; h < NP; h++) cnt[i][j][g][h] += __popc(aw[i][g] & v & bw[j][h]);
        uint32_t ax[PA][NP];
#pragma unroll
        for (int i = 0; i < PA; i++)
#pragma unroll
            for (int g = 0; g < NP; g++) ax[i][g] = aw[i][g];
        if (w + 1 < P.nw) words(w + 1);
        // the rows of individual k + DEPTH are read while those of k are used (three ahead: no faster, one wave less)
        constexpr int DEPTH = 1;
        typename PlainLds<FAST>::row r[DEPTH + 1][PB];
        auto fetch = [&](int k) {
#pragma unroll
            for (int j = 0; j < PB; j++) r[k % (DEPTH + 1)][j] = lds.y[w & 1][k][PB * tx + j];
        };
#pragma unroll
        for (int k = 0; k < DEPTH; k++) fetch(k);
        uint32_t ac[PA][NP];
#pragma unroll
        for (int k = 0; k < 32; k++) {
            if (k % 8 == 0)
#pragma unroll
                for (int i = 0; i < PA; i++)
#pragma unroll
                    for (int g = 0; g < NP; g++) ac[i][g] = k < 24 ? ax[i][g] << (16 - k) : ax[i][g] >> 8;
            if (k + DEPTH < 32) fetch(k + DEPTH);
            const auto &y = r[k % (DEPTH + 1)];
#pragma unroll
            for (int i = 0; i < PA; i++)
#pragma unroll
                for (int g = 0; g < NP; g++) {
                    const float m = __uint_as_float(ac[i][g] & (1u << (16 + k % 8)));
#pragma unroll
                    for (int j = 0; j < PB; j++) {
#pragma unroll
                        for (int h = 0; h < NP; h++) sf[i][j][g][h] = fmaf(m, y[j][h], sf[i][j][g][h]);
                        if (g == 2) qf[i][j] = fmaf(m, y[j][NP], qf[i][j]);
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        // promote the word's FP32 partial sums
#pragma unroll
        for (int i = 0; i < PA; i++)
#pragma unroll
            for (int j = 0; j < PB; j++) {
                if (!FAST) qd[i][j] += (double)qf[i][j];
                qf[i][j] = 0.0f;
#pragma unroll
                for (int g = 0; g < NP; g++)
#pragma unroll
                    for (int h = 0; h < NP; h++) {
                        sd[i][j][g][h] += (double)sf[i][j][g][h];
                        sf[i][j][g][h] = 0.0f;
                    }
            }
        __syncthreads();  // the next word is staged, this one read
    }

#pragma unroll
    for (int i = 0; i < PA; i++) {
        const int a = a0 + PA * ty + i;
        const Marg ma = P.marg[as[i]];
#pragma unroll
        for (int j = 0; j < PB; j++) {
            const int b = b0 + PB * tx + j;
            const Marg mb = P.marg[bs[j]];
            int xc[3][3];
            double xs[3][3];
            double sq;
            if (FAST) {
#pragma unroll
                for (int g = 0; g < 2; g++) {
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        xc[g][h] = cnt[i][j][g][h];
                        xs[g][h] = sd[i][j][g][h] / PLAIN_SCALE;
                    }
                    xc[g][2] = ma.pn[g];
                    xs[g][2] = ma.ys[g];
                    xc[2][g] = mb.pn[g];
                    xs[2][g] = mb.ys[g];
                }
                xc[2][2] = P.nV;
                xs[2][2] = P.ysV;
                sq = P.y2V;
            } else {
#pragma unroll
                for (int g = 0; g < 3; g++)
#pragma unroll
                    for (int h = 0; h < 3; h++) {
                        xc[g][h] = cnt[i][j][g % NP][h % NP];
                        xs[g][h] = sd[i][j][g % NP][h % NP] / PLAIN_SCALE;
                    }
                sq = qd[i][j] / PLAIN_SCALE;
            }
            int n[9];
            double s[9];
            float sf[9];
            cells_from_x(xc, n);
            cells_from_x(xs, s);
#pragma unroll
            for (int c = 0; c < 9; c++) sf[c] = (float)s[c];
            auto exact = [&](double sd[9], double &sqd) {
#pragma unroll
                for (int c = 0; c < 9; c++) sd[c] = s[c];
                sqd = sq;
            };
            const bool valid = a < a1 && b < b1 && a > b;
            finish_pair<DUMP>(hs, dsk, valid, a, b, n, sf, (float)sq, exact, ma.cls, mb.cls);
        }
    }
}

template <int NT, bool FAST, bool DUMP>
__global__ __launch_bounds__(NT, FAST ? 4 : 2) void plain_kernel(const PlainArgs A)
{
    __shared__ PlainLds<FAST> lds;
    const int4 T = A.tiles[xcd_tile(blockIdx.x, A.ntiles)];
    HitSink hs = A.hs;
    hs.tag = A.S.tag;
    plain_tile<NT, FAST, DUMP>(A.S, hs, A.ds, T.x, T.y, T.z, T.w, lds);
}

}  // namespace epi
