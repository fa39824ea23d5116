// Per-dataset preparation kernels: the 2-bit layout A1 (16 genotypes per
// int32, first individual in the most significant bits, right-aligned tail
// word) is decoded once into the operand layouts of the two pair-kernel forms,
// and per-SNP marginals are computed per phenotype.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kern_screen.h"

namespace epi {

// Every second bit of x, from bit 0, packed into the low 16 bits.
__device__ __forceinline__ uint32_t even_bits(uint32_t x)
{
    x &= 0x55555555u;
    x = (x | (x >> 1)) & 0x33333333u;
    x = (x | (x >> 2)) & 0x0F0F0F0Fu;
    x = (x | (x >> 4)) & 0x00FF00FFu;
    return (x | (x >> 8)) & 0xFFFFu;
}

// Class bits of 16 genotypes, bit t = individual t of the packed word, of which the first `have` exist.
__device__ __forceinline__ void class_bits(uint32_t v, int have, uint32_t &c0, uint32_t &c1, uint32_t &nm)
{
    if (have < 16) v = have > 0 ? v << (32 - 2 * have) : 0u;  // the tail word is right-aligned
    const uint32_t r = __brev(v);                              // individual t: high bit at 2t, low bit at 2t + 1
    const uint32_t hi = r, lo = r >> 1, ok = (1u << have) - 1u;
    c0 = even_bits(~(hi | lo)) & ok;
    c1 = even_bits(lo & ~hi) & ok;
    nm = even_bits(~(hi & lo)) & ok;
}

// Class bits of 32 genotypes (two packed words), of which the first `left` exist.
__device__ __forceinline__ void word_bits(uint32_t v0, uint32_t v1, int left, uint32_t b[3])
{
    b[0] = b[1] = b[2] = 0u;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        int have = left - 16 * h;
        have = have < 0 ? 0 : have > 16 ? 16 : have;
        uint32_t x0, x1, xn;
        class_bits(h ? v1 : v0, have, x0, x1, xn);
        b[0] |= x0 << (16 * h);
        b[1] |= x1 << (16 * h);
        b[2] |= xn << (16 * h);
    }
}

constexpr int TR_SNP = 64, TR_WD = 16;  // SNPs and 32-individual words of a workgroup

// Bitplanes [3][Kw][nsnp] of classes 0 and 1 and of the call-present flag, and the counts of the three per SNP
// (added to cnt [3][nsnp]). A workgroup takes 64 SNPs x 16 words: the packed words come in along the individuals (128
// bytes of one SNP per eight lanes), cross in LDS, and the bitplanes go out along the SNPs. Bounded by memory; as one
// thread per SNP and word that decoded its 32 genotypes one by one from strided loads, the transcode and the class
// counts took 1.08 ms at N = 2000, M = 20001; this and order_planes_kernel take 0.02 ms.
__global__ __launch_bounds__(256) void transcode_kernel(const uint32_t *words, int nid, int npack1, int nsnp, int Kw,
                                                        uint32_t *bits, uint32_t *sbits, int *cnt)
{
    __shared__ uint32_t t[TR_SNP][2 * TR_WD + 1];
    __shared__ int c[3][TR_SNP];
    const int s0 = blockIdx.x * TR_SNP, w0 = blockIdx.y * TR_WD, tid = threadIdx.x;
    if (tid < TR_SNP) c[0][tid] = c[1][tid] = c[2][tid] = 0;
    for (int i = tid; i < TR_SNP * 2 * TR_WD; i += 256) {
        const int s = i / (2 * TR_WD), j = i % (2 * TR_WD), g = 2 * w0 + j;
        t[s][j] = s0 + s < nsnp && g < npack1 ? words[(size_t)(s0 + s) * npack1 + g] : 0u;
    }
    __syncthreads();
    const int sl = tid & 63, s = s0 + sl;
    int n[3] = {0, 0, 0};
    for (int k = tid >> 6; k < TR_WD; k += 4) {
        const int wd = w0 + k;
        if (s >= nsnp || wd >= Kw) break;
        uint32_t b[3];
        word_bits(t[sl][2 * k], t[sl][2 * k + 1], nid - 32 * wd, b);
#pragma unroll
        for (int p = 0; p < 3; p++) {
            bits[((size_t)p * Kw + wd) * nsnp + s] = b[p];
            n[p] += __popc(b[p]);
        }
    }
#pragma unroll
    for (int p = 0; p < 3; p++)
        if (n[p]) atomicAdd(&c[p][sl], n[p]);
    // the same words by SNP (0.003 ms of the transcode at N = 2000, M = 20001)
    for (int i = sbits ? tid : TR_SNP * TR_WD; i < TR_SNP * TR_WD; i += 256) {
        const int r = i / TR_WD, k = i % TR_WD, wd = w0 + k;
        if (s0 + r >= nsnp || wd >= Kw) continue;
        uint32_t b[3];
        word_bits(t[r][2 * k], t[r][2 * k + 1], nid - 32 * wd, b);
#pragma unroll
        for (int p = 0; p < 3; p++) sbits[((size_t)p * nsnp + s0 + r) * Kw + wd] = b[p];
    }
    __syncthreads();
    if (tid < TR_SNP && s0 + tid < nsnp)
#pragma unroll
        for (int p = 0; p < 3; p++)
            if (c[p][tid]) atomicAdd(&cnt[(size_t)p * nsnp + s0 + tid], c[p][tid]);
}

// One thread per (four words, SNP): the bitplanes of the two rarest classes and the call-present flag from those of
// classes 0 and 1, for the plain form and the screen; the first row of workgroups also writes cls, the plane -> class map (2 bits each:
// the two rarest classes, then the commonest), and the missing calls.
__global__ __launch_bounds__(256) void order_planes_kernel(const uint32_t *mbits, const int *cnt, int nid, int nsnp, int Kw,
                                                           uint32_t *bits, int32_t *cls, int32_t *miss)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsnp) return;
    const int n0 = cnt[s], n1 = cnt[nsnp + s], nm = cnt[2 * (size_t)nsnp + s], n2 = nm - n0 - n1;
    int big = 0, nb = n0;
    if (n1 > nb) big = 1, nb = n1;
    if (n2 > nb) big = 2;
    const int p0 = big == 0 ? 1 : 0, p1 = big == 2 ? 1 : 2;
    if (blockIdx.y == 0) {
        cls[s] = p0 | (p1 << 2) | (big << 4);
        miss[s] = nid - nm;
    }
    for (int wd = 4 * blockIdx.y; wd < Kw && wd < 4 * (int)blockIdx.y + 4; wd++) {
        const size_t o = (size_t)wd * nsnp + s, plane = (size_t)Kw * nsnp;
        const uint32_t b0 = mbits[o], b1 = mbits[plane + o], bn = mbits[2 * plane + o], b2 = bn & ~b0 & ~b1;
        bits[o] = p0 == 0 ? b0 : b1;
        bits[plane + o] = p1 == 1 ? b1 : b2;
        bits[2 * plane + o] = bn;
    }
}

// Per SNP, over individuals with a call and a present phenotype: counts and
// phenotype sums of genotype classes 0, 1 and of all calls (NM), stored per
// class for the MFMA form and per bitplane (cls order) for the plain form.
// One workgroup per 64 SNPs: lane = SNP (coalesced bitplane loads), four
// waves split the words and are reduced in LDS. The integer sums are 4 x 8-bit dot products of byte masks with
// the limbs of q and z and the digits of v (the wave's, scalar loads), the sum of the plain form's FP32
// phenotype an FP64 FMA with 0 or 1 per class. Bounded by its VALU work, 20 instructions per individual
// and 64 SNPs: 0.045 ms at N = 2000, M = 20001 (0.10 ms with each value masked and added by itself,
// 0.22 ms as a loop over each lane's own set bits, with gathered loads).
__global__ __launch_bounds__(256) void marginals_kernel(const uint32_t *mbits, int Kw, int nsnp,
                                                        const uint32_t *vbits, const float *yc,
                                                        const int32_t *cls, const int8_t *wts, const int8_t *cw,
                                                        Marg *marg, ScrMarg *smarg)
{
    __shared__ long long sq[4][3][64];
    __shared__ double sy[4][3][64];
    __shared__ int sn[4][3][64];
    __shared__ long long sz[4][64];
    __shared__ int sv[4][2][3][64];
    const int sl = threadIdx.x & 63, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s = blockIdx.x * 64 + sl, sc = s < nsnp ? s : nsnp - 1, Kp = 32 * Kw;
    int n[3] = {0, 0, 0};
    int t[3][6] = {}, tz[4] = {};  // limbs of q, v of one digit, digits of v of two; limbs of z (below 2^28)
    double y[3] = {0.0, 0.0, 0.0};
    for (int wd = grp; wd < Kw; wd += 4) {
        const uint32_t v = vbits[wd];
        const uint32_t b0 = mbits[((size_t)0 * Kw + wd) * nsnp + sc] & v;
        const uint32_t b1 = mbits[((size_t)1 * Kw + wd) * nsnp + sc] & v;
        const uint32_t bn = mbits[((size_t)2 * Kw + wd) * nsnp + sc] & v;
        const uint32_t m[3] = {b0, b1, bn & ~b0 & ~b1};
#pragma unroll
        for (int c = 0; c < 3; c++) n[c] += __popc(m[c]);
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {  // 16 individuals
            const int8_t *wp = wts + 32 * wd + 16 * hf, *cp = cw + 32 * wd + 16 * hf;
            v4i e[3];
#pragma unroll
            for (int c = 0; c < 3; c++) e[c] = expand16<false>((m[c] >> (16 * hf)) & 0xFFFFu);
#pragma unroll
            for (int l = 0; l < 6; l++) {
                const v4i w = *reinterpret_cast<const v4i *>(l < 3 ? wp + (size_t)(1 + l) * Kp : cp + (size_t)(l - 3) * Kp);
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int c = 0; c < 3; c++) t[c][l] = __builtin_amdgcn_sdot4(e[c][k], w[k], t[c][l], false);
            }
            const v4i en = e[0] | e[1] | e[2];
#pragma unroll
            for (int l = 0; l < 4; l++) {
                const v4i w = *reinterpret_cast<const v4i *>(wp + (size_t)(4 + l) * Kp);
#pragma unroll
                for (int k = 0; k < 4; k++) tz[l] = __builtin_amdgcn_sdot4(en[k], w[k], tz[l], false);
            }
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const double yd = (double)yc[32 * wd + 16 * hf + j];
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    int k = __builtin_amdgcn_sbfe((int)m[c], 16 * hf + j, 1);
                    asm("" : "+v"(k));  // kept a mask (a compare and a select otherwise)
                    y[c] = __builtin_fma(__hiloint2double(k & 0x3FF00000, 0), yd, y[c]);
                }
            }
        }
    }
    long long q[3], z;
    int v3[2][3];  // sums of the screen's coarse phenotypes (their magnitude stays below 2^24)
#pragma unroll
    for (int c = 0; c < 3; c++) {
        q[c] = (long long)t[c][0] + 256ll * t[c][1] + 65536ll * t[c][2];
        v3[0][c] = t[c][3];
        v3[1][c] = t[c][4] + 256 * t[c][5];
    }
    z = (long long)tz[0] + 256ll * tz[1] + 65536ll * tz[2] + 16777216ll * tz[3];
    for (int c = 0; c < 3; c++) {
        sn[grp][c][sl] = n[c];
        sq[grp][c][sl] = q[c];
        sy[grp][c][sl] = y[c];
    }
    sz[grp][sl] = z;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int c = 0; c < 3; c++) sv[grp][i][c][sl] = v3[i][c];
    __syncthreads();
    if (grp == 0 && s < nsnp) {
        int tn[3];
        long long tq[3];
        double ty[3];
        for (int c = 0; c < 3; c++) {
            tn[c] = sn[0][c][sl] + sn[1][c][sl] + sn[2][c][sl] + sn[3][c][sl];
            tq[c] = sq[0][c][sl] + sq[1][c][sl] + sq[2][c][sl] + sq[3][c][sl];
            ty[c] = ((sy[0][c][sl] + sy[1][c][sl]) + sy[2][c][sl]) + sy[3][c][sl];
        }
        Marg mg;
        const int cl = cls[s];
        const int ntot = tn[0] + tn[1] + tn[2];
        mg.n[0] = tn[0];
        mg.n[1] = tn[1];
        mg.n[2] = ntot;
        mg.q[0] = tq[0];
        mg.q[1] = tq[1];
        mg.q[2] = tq[0] + tq[1] + tq[2];
        for (int p = 0; p < 2; p++) {
            int c = (cl >> (2 * p)) & 3;
            mg.pn[p] = tn[c];
            mg.ys[p] = ty[c];
        }
        mg.pn[2] = ntot;
        mg.ys[2] = ty[0] + ty[1] + ty[2];
        mg.cls = cl;
        mg.pad = 0;
        mg.zs = sz[0][sl] + sz[1][sl] + sz[2][sl] + sz[3][sl];
        marg[s] = mg;
        const float u = 1.0f / 64.0f;
        ScrMarg sm;
        for (int p = 0; p < 3; p++) {
            const int c = (cl >> (2 * p)) & 3;
            sm.n[p] = (float)tn[c] * u;
            for (int i = 0; i < 2; i++)
                sm.s[i][p] = (float)(sv[0][i][c][sl] + sv[1][i][c][sl] + sv[2][i][c][sl] + sv[3][i][c][sl]) * u;
        }
        sm.zs = (float)mg.zs;
        sm.s[0][3] = sm.s[1][3] = 0.0f;
        smarg[s] = sm;
    }
}

// Codes of one phenotype's outlier individuals per SNP (thread = SNP): two
// bits per outlier, the genotype class (0, 1, 2) or 3 for a missing call;
// word w holds outliers 16w..16w+15, stored [w][snp] so that a wave's SNPs
// read consecutive words.
__global__ __launch_bounds__(256) void outlier_codes_kernel(const uint32_t *mbits, int Kw, int nsnp,
                                                            const int32_t *oidx, int nout, uint32_t *ocodes)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsnp) return;
    for (int w = 0; 16 * w < nout; w++) {
        uint32_t code = 0;
        for (int t = 0; t < 16 && 16 * w + t < nout; t++) {
            const int k = oidx[16 * w + t], wd = k >> 5;
            const uint32_t bit = 1u << (k & 31);
            const bool c0 = (mbits[((size_t)0 * Kw + wd) * nsnp + s] & bit) != 0;
            const bool c1 = (mbits[((size_t)1 * Kw + wd) * nsnp + s] & bit) != 0;
            const bool nm = (mbits[((size_t)2 * Kw + wd) * nsnp + s] & bit) != 0;
            const uint32_t g = !nm ? 3u : c0 ? 0u : c1 ? 1u : 2u;
            code |= g << (2 * t);
        }
        ocodes[(size_t)w * nsnp + s] = code;
    }
}

// One thread per SNP: the individuals (below nid) without a call, ascending,
// into mlist[moff[s] ...].
__global__ __launch_bounds__(256) void miss_list_kernel(const uint32_t *mbits, int Kw, int nsnp, int nid,
                                                        const long long *moff, int32_t *mlist)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsnp) return;
    long long o = moff[s];
    for (int wd = 0; wd < Kw && 32 * wd < nid; wd++) {
        uint32_t x = ~mbits[((size_t)2 * Kw + wd) * nsnp + s];
        if (nid - 32 * wd < 32) x &= (1u << (nid - 32 * wd)) - 1u;
        while (x) {
            mlist[o++] = 32 * wd + __ffs(x) - 1;
            x &= x - 1u;
        }
    }
}

// Transposed bitplanes for the SPARSE tiles: one wave per (64-SNP word wv of
// the virtual SNP order, 32-individual word wd). Lane l is virtual SNP
// 64 wv + l (snp_of_v: its SNP, or -1 for padding); a ballot over the lanes
// of bit k of a plane word is the 64-SNP word of individual 32 wd + k, which
// lane k collects and stores: tbits[wv][32 wd + k][plane], planes class 0,
// class 1, call present, and a zero word (a 64-SNP column is contiguous).
__global__ __launch_bounds__(64) void tbits_kernel(const uint32_t *mbits, int Kw, int nsnp, int nid,
                                                    const int32_t *snp_of_v, int nw, uint64_t *tbits)
{
    const int wv = blockIdx.x, wd = blockIdx.y, l = threadIdx.x;
    const int s = snp_of_v[64 * wv + l];
    uint32_t lo[3] = {0u, 0u, 0u}, hi[3] = {0u, 0u, 0u};
#pragma unroll
    for (int p = 0; p < 3; p++) {
        const uint32_t x = s >= 0 ? mbits[((size_t)p * Kw + wd) * nsnp + s] : 0u;
        for (int k = 0; k < 32; k++) {
            const uint64_t b = __ballot((x >> k) & 1u);
            lo[p] = l == k ? (uint32_t)b : lo[p];
            hi[p] = l == k ? (uint32_t)(b >> 32) : hi[p];
        }
    }
    const int i = 32 * wd + l;
    if (l < 32 && i < nid) {
        uint64_t *o = tbits + ((size_t)wv * nid + i) * 4;
#pragma unroll
        for (int p = 0; p < 3; p++) o[p] = ((uint64_t)hi[p] << 32) | lo[p];
        o[3] = 0ull;
    }
}

}  // namespace epi
