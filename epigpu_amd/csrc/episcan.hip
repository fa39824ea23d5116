// libepiscan.so - C ABI over the MI355X (gfx950) pair-scan kernels.
//
// Device state of one dataset (a context holds one; a batch holds many):
//   words   [nsnp][npack1] int32   genotypes as uploaded (layout A1), freed after the transcode
//   mbits   [3][Kw][nsnp]  uint32  bitplanes of classes 0, 1 and call present (MFMA form)
//   sbits   [3][nsnp][Kw]  uint32  the same by SNP (resolve kernel), or null: given back where memory is short
//   bits    [3][Kw][nsnp]  uint32  bitplanes of the two rarest classes and call present (plain form)
//   cls     [nsnp]         int32   plain-form plane -> class map
//   per phenotype r (wts, mp, yc, yw, vbits, ov and oidx in one allocation):
//     wts   [8][Kp] int8   V, 3 limbs of q, 4 limbs of round(q^2/2^zbits)
//     yc    [Kp]    float  centred phenotype scaled by 2^-ybits to |yc| < 1 (0 where missing)
//     yw    [2][Kp] float  yc and its square as the plain kernel reads them
//     vbits [Kw]    uint32 phenotype-present bits
//     marg  [nsnp]  Marg   per-SNP class counts and sums
//     oidx, ocodes, ov     outlier individuals (at most OUT_MAX), their codes per SNP and values
//     mp    [Kp]    MissPhen V, q, z per individual (SPARSE tiles), coarse phenotype v of the screen
//     sw    [Kw][8], [Kw][16] uint32  the screen's FP6 codes of v (one and two digits) and presence bits, per
//                   32 individuals (behind wts), then [3][Kp] int8, v in base-256 digits (marginals)
//     sm    [nsnp]  ScrMarg per-SNP counts and sums of v (before marg, in its allocation)
//   for SPARSE tiles (built at the first scan that has them, for the chromosome layout it was built for):
//     moff  [nsnp+1] int64, mlist int32   per SNP, the individuals with a missing call
//     vidx  [nsnp]  int32  virtual SNP index: each chromosome starts at a multiple of 64
//     tbits [nw][nid][4] uint64  transposed bitplanes over the virtual order (64 SNPs per word)
// Kp = nid rounded up to 256 (the plain kernel's stage), Kw = Kp / 32; padding
// individuals are absent. The MFMA K loops stop at nid rounded up to 128.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "episcan.h"
#include "kern_batch.h"
#include "kern_mfma.h"
#include "kern_plain.h"
#include "kern_screen.h"
#include "transcode.h"

using namespace epi;

namespace {

constexpr int KPAD = 256;
// The grid of tbits_kernel has one row of workgroups per 32 individuals, and a
// grid row index stays below 65536: at most 8191 K-pads of individuals.
constexpr int MAX_NID = 65535 / (KPAD / 32) * KPAD;
constexpr long long QMAX = 8355711;     // largest |q| with three balanced int8 limbs
constexpr long long ZMAX = 2139062143;  // largest |z| with four balanced int8 limbs
// The MFMA form's phenotype range. The central SD s_c is the SD of the
// present values without the 2 OUT_MAX farthest from the median (a quarter of
// them when there are fewer than 258). Among the OUT_MAX farthest, values more
// than OUT_SD s_c from the central mean are outliers, carried exactly. The
// encoded values must then lie within BULK_SD s_c of the centre, which bounds
// the fixed-point quantum at BULK_SD / QMAX = 7.7e-6 s_c; a phenotype beyond
// that is refused by MFMA scans (EPI_ERR_RANGE), and the plain form, FP32 per
// value, takes it.
constexpr double OUT_SD = 32.0;
constexpr double BULK_SD = 64.0;

// The coarse phenotype of the screen, of one or two digits: q ~ delta v + offset.
struct ScreenEnc {
    double delta = 0.0;   // 0: none
    double offset = 0.0;
    double eps = 0.0;     // |q - delta v - offset| over the present individuals
    double vsum = 0.0;    // sum of v
};

struct PhenDev {
    int8_t *wts = nullptr;
    float *yc = nullptr;
    float *yw = nullptr;
    uint32_t *vbits = nullptr;
    Marg *marg = nullptr;
    int32_t *oidx = nullptr;    // [nout] outlier individuals
    uint32_t *ocodes = nullptr; // [ceil(nout/16)][nsnp], built with the marginals
    OutVals *ov = nullptr;
    MissPhen *mp = nullptr;
    uint32_t *sw[2] = {nullptr, nullptr};  // screen (in the allocation of wts)
    ScrMarg *sm = nullptr;                 // screen (owns marg)
    ScreenEnc scr[2];
    double zall = 0.0;          // sum of z
    int nout = 0;
    int fbits = 0;  // q = round((y - centre) * 2^fbits)
    int zbits = 0;  // Z limbs hold round(q^2 / 2^zbits)
    int ybits = 0;  // plain form: yc = (y - centre) * 2^-ybits, |yc| < 1
    double centre = 0.0;
    int nV = 0;
    long long qV = 0;
    double sqV = 0.0;  // sum q^2
    double ysV = 0.0;  // sum yc
    double y2V = 0.0;  // sum yc^2
    double ouSum = 0.0, ouSq = 0.0;  // sum of the outliers' values (units 2^-fbits) and of their squares
    double sc = 0.0, maxdev = 0.0;   // central SD; largest |y - centre| of the encoded values
    bool mfma_ok = true;
    std::string mfma_why;
};

struct Dataset {
    int nid = 0, nsnp = 0, npack1 = 0, Kp = 0, Kw = 0;
    int32_t *words = nullptr;
    uint32_t *mbits = nullptr;
    uint32_t *sbits = nullptr;
    uint32_t *bits = nullptr;
    int32_t *dmiss = nullptr;
    int32_t *cls = nullptr;
    std::vector<int> miss;    // per SNP: missing calls
    std::vector<int> missc;   // prefix count of SNPs with missing calls
    std::vector<int> heavyc;  // prefix count of SNPs with more than sparse_max() missing calls
    std::vector<long long> missum;  // prefix sum of missing calls
    std::vector<PhenDev> ph;
    bool marg_ok = false;
    std::vector<int> chrstart, chrsize, snpchr;
    // SPARSE tiles
    bool sp_ok = false;       // built for the current genotypes and chromosomes
    long long *moff = nullptr;
    int32_t *mlist = nullptr;
    int32_t *vidx = nullptr;
    uint64_t *tbits = nullptr;
    long long tstride = 0;    // uint64 words per 64-SNP column of tbits (4 nid)
};

// Tile lists of a scan by kind: FAST (no missing call), SPARSE (missing
// calls, few per SNP), GENERAL (the rest). Device order: FAST, SPARSE, GENERAL.
struct TileLists {
    std::vector<int4> fast, gen, sp;
    long long pairs = 0;
    size_t count() const { return fast.size() + sp.size() + gen.size(); }
};

}  // namespace

struct epi_ctx {
    int device = 0;
    int ncu = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::string err;
    char name[256] = {0};
    Dataset d;
    std::vector<epi_batch *> batches;
    // hits
    DevHit *hits = nullptr;
    long long cap = 1ll << 22;
    long long last_nhits = 0;
    // counters of the hits and of the screen; candidates; blocks to redo and their masks (behind the tiles, or null)
    Counters *count = nullptr;
    int4 *cand = nullptr;
    uint32_t *redo = nullptr;
    size_t redo_blocks = 0;
    bool masks_set = false;  // cleared since the list was built
    // tiles; the device list of the last scan is kept and reused while the
    // dataset, block range, form and schedule stay the same
    int4 *tiles = nullptr;
    size_t tiles_cap = 0;
    size_t max_tiles = (size_t)1 << 25;  // 512 MiB of int4
    TileLists tl;
    bool tl_valid = false;
    int tl_bb = 0, tl_be = 0, tl_form = -1;
    epi_schedule tl_sched = {};
    // stats
    double last_ms = 0.0;
    long long last_pairs = 0;
    int last_launches = 0;
    long long last_tiles[3] = {0, 0, 0};  // FAST, SPARSE, GENERAL tiles of the last scan
    int last_digits = 0;                  // of the screen in the last scan; 0: not screened
    long long last_cand = 0, last_redone = 0;
    epi_schedule sched[2];  // per form
    void *scratch = nullptr;  // this device's no-allocation scratch (address from hipGetSymbolAddress)
};

struct epi_batch {
    epi_ctx *ctx = nullptr;
    std::vector<Dataset *> data;
    std::vector<std::pair<int, int>> scans;  // (dataset, phenotype)
    MfmaScan *d_mscan = nullptr;
    PlainScan *d_pscan = nullptr;
    ScreenCut *d_cut = nullptr;
    uint32_t *redo = nullptr, *mask = nullptr;  // behind the work items
    int4 *d_work = nullptr;
    int *d_qpos = nullptr, *d_qbegin = nullptr, *d_qend = nullptr;  // [NLIST][NQ]
    size_t work_cap = 0, scan_cap = 0;
    long long nlist[NLIST] = {};  // work items of each list (in this order in d_work)
    std::vector<std::pair<int, long long>> segs[NKIND];  // the datasets of a screened list, in its order, and their items
    DevHit *hits = nullptr;
    Counters *count = nullptr;
    long long cap = 1ll << 22;
    // work list of the last build
    epi_schedule sched[2];  // per form
    epi_schedule work_sched = {};
    std::vector<char> work_scr;  // the scans that are screened
    int scr_rows = 0;            // tile height of their lists
    bool dirty = true;
    int work_form = -1;
    long long nwork = 0, pairs = 0;
    // captured graph of the last scan
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    epi_scan_params gkey = {};
    bool gvalid = false;
    int captures = 0;
    int grid = 0;
    // results
    long long last_nhits = 0;
    double last_ms = 0.0;
    int gscreened = 0;  // scans that the captured graph screens
    int last_screened = 0;
    long long last_cand = 0, last_redone = 0;
    bool fetched = false;
    std::vector<DevHit> hh;
    std::vector<std::vector<int>> by_scan;
};

namespace {

int fail(epi_ctx *c, int code, const char *fmt, ...)
{
    if (c) {
        char buf[512];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        c->err = buf;
    }
    return code;
}

#define HIPCHK(c, call)                                                                          \
    do {                                                                                         \
        hipError_t e_ = (call);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return fail((c), EPI_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                        __FILE__, __LINE__);                                                     \
    } while (0)

template <class T>
void dfree(T *&p)
{
    if (p) (void)hipFree(p);
    p = nullptr;
}

bool give_back(epi_ctx *c);

template <class T>
int dalloc(epi_ctx *c, T *&p, size_t count)
{
    dfree(p);
    if (count == 0) count = 1;
    hipError_t e = hipMalloc((void **)&p, count * sizeof(T));
    if (e != hipSuccess && give_back(c)) {
        (void)hipGetLastError();
        e = hipMalloc((void **)&p, count * sizeof(T));
    }
    if (e != hipSuccess) {
        p = nullptr;
        (void)hipGetLastError();  // not to be found after a later launch
        return fail(c, EPI_ERR_NOMEM, "hipMalloc of %zu bytes failed: %s", count * sizeof(T), hipGetErrorString(e));
    }
    return EPI_OK;
}

void free_phen(PhenDev &p)
{
    dfree(p.wts);  // with the arrays behind it
    p.sw[0] = p.sw[1] = nullptr;
    p.mp = nullptr;
    p.yc = nullptr;
    p.yw = nullptr;
    p.vbits = nullptr;
    p.ov = nullptr;
    p.oidx = nullptr;
    dfree(p.sm);
    p.marg = nullptr;
    dfree(p.ocodes);
}

void drop_sparse(Dataset &d)
{
    dfree(d.moff);
    dfree(d.mlist);
    dfree(d.vidx);
    dfree(d.tbits);
    d.sp_ok = false;
}

void drop_phenotypes(Dataset &d)
{
    for (auto &p : d.ph) free_phen(p);
    d.ph.clear();
    d.marg_ok = false;
}

void free_dataset(Dataset &d)
{
    dfree(d.words);
    dfree(d.mbits);  // with the arrays behind it
    d.bits = nullptr;
    d.dmiss = d.cls = nullptr;
    dfree(d.sbits);
    drop_sparse(d);
    for (auto &p : d.ph) free_phen(p);
    d.ph.clear();
}

// The bits by SNP of every dataset of the context, which scans can do without, to an allocation that failed.
// Whether there were any. The batches' descriptors point to them and are built again.
bool give_back(epi_ctx *c)
{
    if (!c) return false;
    bool any = c->d.sbits != nullptr;
    for (epi_batch *b : c->batches)
        for (Dataset *d : b->data) any |= d->sbits != nullptr;
    if (!any) return false;
    (void)hipStreamSynchronize(c->stream);
    dfree(c->d.sbits);
    for (epi_batch *b : c->batches)
        for (Dataset *d : b->data) {
            if (d->sbits) b->dirty = true;
            dfree(d->sbits);
        }
    return true;
}

// ------------------------------------------------------ dataset preparation --

// SNPs with at most this many missing calls can be in SPARSE tiles (the
// per-pair counts of the missing-call sums are 16-bit).
int sparse_max(int nid) { return std::min(65535, std::max(8, nid / 16)); }

// A tile with missing calls is SPARSE (under dense_missing 0) when its SNPs
// miss at most 1 / SPARSE_RATE of their calls on average: measured at
// N = 4000 with 64-row tiles, the per-individual sums of a SPARSE tile cost
// less than the NM rows of a GENERAL tile up to about 0.7 % missing calls
// (0.5 %: 17.7 ms against 20.5 ms for the scan; 1 %: 24.7 against 20.5).
constexpr long long SPARSE_RATE = 150;

// Two bitplanes below 4 GiB, as the screen's buffer descriptors take them.
bool planes_fit(const Dataset &d) { return (unsigned long long)d.Kw * d.nsnp * 8ull < (1ull << 32) - (1u << 20); }

int ds_upload_genotypes(epi_ctx *c, Dataset &d, const int32_t *words, int nid, int nsnp)
{
    if (!d.ph.empty() && nid != d.nid) drop_phenotypes(d);  // a new cohort: the old phenotypes no longer apply
    drop_sparse(d);
    d.nid = nid;
    d.nsnp = nsnp;
    d.npack1 = (nid + 15) / 16;
    d.Kp = (nid + KPAD - 1) / KPAD * KPAD;
    d.Kw = d.Kp / 32;
    size_t nwords = (size_t)nsnp * d.npack1;
    int rc;
    // one allocation for what the dataset keeps: bitplanes, bits, dmiss, cls, each on a 256-byte boundary
    const size_t planes = (size_t)3 * d.Kw * nsnp, room = (planes + 63) / 64 * 64, per = ((size_t)4 * nsnp + 63) / 64 * 64;
    if ((rc = dalloc(c, d.mbits, 2 * room + per + nsnp)) || (rc = dalloc(c, d.words, nwords))) return rc;
    d.bits = d.mbits + room;
    d.dmiss = reinterpret_cast<int32_t *>(d.bits + room);
    d.cls = d.dmiss + per;
    // Bits by SNP, where the screen can run and memory allows: the lanes of the resolve kernel, one word each,
    // then read a SNP's words in a row (N = 3001, 67,000 hits: resolve 250 -> 156 us; N = 2000: 84 -> 42 us). Allocated last, and
    // given back to whatever finds no memory (give_back). The old ones are freed here and not first, so that the new ones find their
    // place: loading another dataset of N = 4000, M = 20000 takes 1.01 and not 1.25 ms.
    dfree(d.sbits);
    if (planes_fit(d) && hipMalloc((void **)&d.sbits, planes * sizeof(uint32_t)) != hipSuccess) {
        d.sbits = nullptr;
        (void)hipGetLastError();
    }
    HIPCHK(c, hipMemcpyAsync(d.words, words, nwords * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    int *cnt = d.dmiss + nsnp;  // class counts of the SNPs
    HIPCHK(c, hipMemsetAsync(cnt, 0, 3 * (size_t)nsnp * sizeof(int), c->stream));
    hipLaunchKernelGGL(transcode_kernel, dim3((nsnp + TR_SNP - 1) / TR_SNP, (d.Kw + TR_WD - 1) / TR_WD), dim3(256), 0,
                       c->stream, (const uint32_t *)d.words, nid, d.npack1, nsnp, d.Kw, d.mbits, d.sbits,
                       cnt);
    HIPCHK(c, hipGetLastError());
    hipLaunchKernelGGL(order_planes_kernel, dim3((nsnp + 255) / 256, (d.Kw + 3) / 4), dim3(256), 0, c->stream,
                       (const uint32_t *)d.mbits, (const int *)cnt, nid, nsnp, d.Kw, d.bits, d.cls, d.dmiss);
    HIPCHK(c, hipGetLastError());
    d.miss.assign(nsnp, 0);
    HIPCHK(c, hipMemcpyAsync(d.miss.data(), d.dmiss, (size_t)nsnp * sizeof(int32_t), hipMemcpyDeviceToHost,
                             c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    dfree(d.words);  // the uploaded words only feed the transcode
    d.missc.assign(nsnp + 1, 0);
    d.heavyc.assign(nsnp + 1, 0);
    d.missum.assign(nsnp + 1, 0);
    const int smax = sparse_max(nid);
    for (int s = 0; s < nsnp; s++) {
        d.missc[s + 1] = d.missc[s] + (d.miss[s] != 0);
        d.heavyc[s + 1] = d.heavyc[s] + (d.miss[s] > smax);
        d.missum[s + 1] = d.missum[s] + d.miss[s];
    }
    d.marg_ok = false;
    // chromosome layout resets to one block over all SNPs
    d.chrstart.assign(1, 0);
    d.chrsize.assign(1, nsnp);
    d.snpchr.assign(nsnp, 0);
    return EPI_OK;
}

// New genotypes. A failure after the arguments are checked leaves the
// dataset empty (genotypes and phenotypes unset), never half updated.
int ds_set_genotypes(epi_ctx *c, Dataset &d, const int32_t *words, int nid, int nsnp)
{
    if (!words || nid < 2 || nsnp < 2) return fail(c, EPI_ERR_ARG, "need nid >= 2, nsnp >= 2 and words");
    if (nid > MAX_NID) return fail(c, EPI_ERR_RANGE, "nid %d above the supported %d", nid, MAX_NID);
    d.marg_ok = false;
    const int rc = ds_upload_genotypes(c, d, words, nid, nsnp);
    if (rc) {
        free_dataset(d);
        d = Dataset();
    }
    return rc;
}

// Balanced signed 8-bit limbs of x, least significant first; false if x needs more than n.
bool split_limbs(long long x, int n, int8_t *out)
{
    for (int i = 0; i < n; i++) {
        const long long l = ((x % 256) + 256 + 128) % 256 - 128;
        out[i] = (int8_t)l;
        x = (x - l) / 256;
    }
    return x == 0;
}

// Host-side encoding of one phenotype, before anything is allocated.
struct PhenEnc {
    std::vector<int8_t> w;      // [NWP][Kp], then the screen's weights (3 Kp bytes) and [NWC][Kp]
    std::vector<int32_t> qv;    // [Kp]
    std::vector<float> yc;      // [Kp]
    std::vector<float> yw;      // [2][Kp]
    std::vector<uint32_t> vb;   // [Kw]
    std::vector<int32_t> oidx;  // outlier individuals
    std::vector<MissPhen> mp;   // [Kp]
    OutVals ov = {};
    PhenDev p;                  // scalars only
};

// Coarse phenotypes of the screen. A digit is an integer that FP6 E2M3 holds in
// units of 1/8: 0..16, even to 30, multiples of 4 to 60, either sign.
constexpr int SCR_VMAX1 = 60, SCR_VMAX2 = 32 * 60 + 60;

uint32_t fp6_code(int d)
{
    const int a = std::abs(d);
    const uint32_t c = a < 16 ? (uint32_t)a : a < 32 ? 16u + (uint32_t)(a / 2 - 8) : 24u + (uint32_t)(a / 4 - 8);
    return c | (d < 0 ? 32u : 0u);
}

// Nearest representable v = D0 and v = 32 D1 + D0 of every integer up to the largest, with their codes.
struct ScrTable {
    struct Entry {
        int16_t v;
        uint8_t c0, c1;
    };
    Entry one[2 * SCR_VMAX1 + 1], two[2 * SCR_VMAX2 + 1];
    ScrTable()
    {
        std::vector<int> digit;
        for (int d = -60; d <= 60; d++)
            if (std::abs(d) <= 16 || (std::abs(d) <= 32 && d % 2 == 0) || d % 4 == 0) digit.push_back(d);
        auto fill = [](Entry *t, int vmax) {  // nearest set entries into the gaps
            std::vector<Entry> full(t, t + 2 * vmax + 1);
            for (int i = 0; i <= 2 * vmax; i++)
                for (int o = 0;; o++) {
                    if (i - o >= 0 && full[i - o].v != INT16_MAX) { t[i] = full[i - o]; break; }
                    if (i + o <= 2 * vmax && full[i + o].v != INT16_MAX) { t[i] = full[i + o]; break; }
                }
        };
        for (Entry &e : one) e = {INT16_MAX, 0, 0};
        for (Entry &e : two) e = {INT16_MAX, 0, 0};
        for (int d : digit) one[d + SCR_VMAX1] = {(int16_t)d, (uint8_t)fp6_code(d), 0};
        for (int h : digit)
            for (int l : digit) two[32 * h + l + SCR_VMAX2] = {(int16_t)(32 * h + l), (uint8_t)fp6_code(l), (uint8_t)fp6_code(h)};
        fill(one, SCR_VMAX1);
        fill(two, SCR_VMAX2);
    }
    const Entry &get(int nd, double t) const
    {
        const int m = nd == 1 ? SCR_VMAX1 : SCR_VMAX2;
        const int i = (int)std::lrint(std::min((double)m, std::max((double)-m, t)));
        return (nd == 1 ? one : two)[i + m];
    }
};

const ScrTable &scr_table()
{
    static const ScrTable t;
    return t;
}

// Sums of a fit of q on v.
struct ScrFit {
    double n = 0.0, q = 0.0, v = 0.0, qq = 0.0, qv = 0.0, vv = 0.0, va = 0.0;
    void add(double x, double y)
    {
        n += 1.0;
        q += x;
        v += y;
        qq += x * x;
        qv += x * y;
        vv += y * y;
        va += std::fabs(y);
    }
    // squared residue of the least-squares line
    double residue(double &slope, double &off) const
    {
        const double cvv = vv - v * v / n, cqv = qv - q * v / n;
        slope = cvv > 0.0 ? cqv / cvv : 0.0;
        off = (q - slope * v) / n;
        return std::max(0.0, qq - q * q / n - slope * cqv);
    }
};

// v of nd digits for the present individuals P: q / step, rounded to what the digits hold, then the line q ~ delta v
// + offset of least squares, whose residue is what the bound pays. Two digits: the smallest step without
// clipping. One digit: the best of a few, clipping included, on up to 1024 individuals. The sum of |v|
// stays below 2^24, so that every sum of v in FP32 is exact.
void encode_screen(const std::vector<int> &P, int Kp, int nd, PhenEnc &e)
{
    ScreenEnc &S = e.p.scr[nd - 1];
    S = ScreenEnc();
    const ScrTable &T = scr_table();
    double mx = 0.0, sum = 0.0;
    for (int k : P) {
        const double a = std::fabs((double)e.qv[k]);
        mx = std::max(mx, a);
        sum += a;
    }
    const double room = 16777216.0 - (nd == 1 ? 4.0 : 130.0) * (double)P.size();  // |v| exceeds |q| / step by less
    if (!(mx > 0.0) || room <= 0.0) return;
    const double least = sum / room;
    double step = std::max(mx / (nd == 1 ? SCR_VMAX1 : SCR_VMAX2), least), slope, off;
    if (nd == 1) {
        const size_t stride = (P.size() + 1023) / 1024;
        double best = INFINITY, top = step;
        for (double f : {1.0, 0.8, 0.65, 0.5, 0.4}) {
            ScrFit F;
            for (size_t i = 0; i < P.size(); i += stride) F.add(e.qv[P[i]], T.get(1, e.qv[P[i]] / (f * top)).v);
            const double r = F.residue(slope, off);
            if (f * top >= least && slope > 0.0 && r < best) {
                best = r;
                step = f * top;
            }
        }
    }
    ScrFit F;
    const double inv = 1.0 / step;
    uint32_t *rows = reinterpret_cast<uint32_t *>(e.w.data() + (size_t)NWP * Kp) + (nd == 1 ? 0 : Kp / 4);
    const int row = 8 * nd;
    for (int k : P) {
        const ScrTable::Entry &t = T.get(nd, e.qv[k] * inv);
        e.mp[k].sv[nd - 1] = t.v;
        F.add(e.qv[k], t.v);
        // the element of individual k & 31: six bits from bit 6 slot of the word's 192
        static const struct Slots {
            int bit[32];
            Slots() { for (int i = 0; i < 32; i++) bit[i] = 6 * scr_slot(i); }
        } slots;
        const int bit = slots.bit[k & 31];
        uint32_t *r = rows + (size_t)(k >> 5) * row;
        for (int i = 0; i < nd; i++) {
            const uint64_t c = (uint64_t)(i ? t.c1 : t.c0) << (bit & 31);
            r[6 * i + (bit >> 5)] |= (uint32_t)c;
            if (c >> 32) r[6 * i + (bit >> 5) + 1] |= (uint32_t)(c >> 32);
        }
        r[6 * nd] |= 1u << (k & 31);
    }
    const double r2 = F.residue(slope, off);
    if (!(slope > 0.0) || F.va >= 16777216.0) return;
    S.delta = slope;
    S.offset = off;
    // (the residue is a difference of sums of N terms: their rounding is added)
    S.eps = std::sqrt(r2 + 1e-12 * F.qq) * (1.0 + 1e-6);
    S.vsum = F.v;
}

// Phenotype prep (src/EpiOpenCL.c:1364-1376 computes mY and SSY over all nid
// and the kernel drops -9 values, :135-147; here the missing values are
// dropped up front). Centre, outliers and fixed-point scale of the MFMA
// form, the plain form's scaled FP32 values, presence bits, the coarse phenotypes of the screen; without `arrays` only
// what epi_phen_encoding reports.
int encode_phen(epi_ctx *c, const float *y, int nid, int Kp, bool nine_value, int r, bool arrays, PhenEnc &e)
{
    auto missing = [&](float v) { return v != v || (!nine_value && v == -9.0f); };
    std::vector<int> P;
    P.reserve(nid);
    for (int k = 0; k < nid; k++) {
        const float v = y[k];
        if (missing(v)) continue;
        if (std::isinf(v)) return fail(c, EPI_ERR_RANGE, "phenotype %d has an infinite value", r);
        P.push_back(k);
    }
    const int nv = (int)P.size();
    if (nv < 2) return fail(c, EPI_ERR_RANGE, "phenotype %d has fewer than 2 present values", r);
    PhenDev &p = e.p;
    // Outliers among the ntop values farthest from the median (which far values
    // cannot drag), measured against the central values (all but the ncen farthest).
    std::vector<float> med(nv);
    for (int t = 0; t < nv; t++) med[t] = y[P[t]];
    std::nth_element(med.begin(), med.begin() + nv / 2, med.end());
    const double c0 = (double)med[nv / 2];
    const int ncen = std::min(2 * OUT_MAX, (nv - 2) / 4), ntop = std::min(OUT_MAX, ncen);
    std::vector<int> ord(P);
    auto farther = [&](int x, int z) {
        const double dx = std::fabs((double)y[x] - c0), dz = std::fabs((double)y[z] - c0);
        return dx != dz ? dx > dz : x < z;
    };
    if (ncen > 0) {
        std::nth_element(ord.begin(), ord.begin() + ncen - 1, ord.end(), farther);
        std::sort(ord.begin(), ord.begin() + ncen, farther);
    }
    std::vector<char> far(nid, 0), out(nid, 0);
    for (int t = 0; t < ncen; t++) far[ord[t]] = 1;
    double mb = 0.0, sb = 0.0;
    for (int k : P)
        if (!far[k]) mb += (double)y[k];
    mb /= (nv - ncen);
    for (int k : P)
        if (!far[k]) sb += ((double)y[k] - mb) * ((double)y[k] - mb);
    sb = std::sqrt(sb / (nv - ncen));
    for (int t = 0; t < ntop; t++) {
        const int k = ord[t];
        if (std::fabs((double)y[k] - mb) > OUT_SD * sb) {
            out[k] = 1;
            e.oidx.push_back(k);
        }
    }
    p.nout = (int)e.oidx.size();
    double centre = 0.0;
    for (int k : P)
        if (!out[k]) centre += (double)y[k];
    centre /= (nv - p.nout);
    double maxabs = 0.0, maxall = 0.0;
    for (int k : P) {
        const double dv = std::fabs((double)y[k] - centre);
        maxall = std::max(maxall, dv);
        if (!out[k]) maxabs = std::max(maxabs, dv);
    }
    p.sc = sb;
    p.maxdev = maxabs;
    p.mfma_ok = maxabs <= BULK_SD * sb;
    if (!p.mfma_ok) {
        char buf[256];
        snprintf(buf, sizeof(buf),
                 "phenotype %d: more than %d values lie far out (after %d outliers, a value %.3g central SDs "
                 "out remains, above %g); the MFMA form's fixed point cannot hold it to 1e-5, use the plain form",
                 r, OUT_MAX, p.nout, sb > 0.0 ? maxabs / sb : INFINITY, BULK_SD);
        p.mfma_why = buf;
    }
    int f = 0;
    if (maxabs > 0.0) f = (int)std::floor(std::log2((double)QMAX / maxabs));
    while (maxabs > 0.0 && std::ldexp(maxabs, f) > (double)QMAX) f--;
    // the plain form's FP32 values are scaled by a power of two to |yc| < 1, so that products of
    // phenotypes far from unit scale neither overflow nor underflow FP32 (F is scale-free)
    int ye = 0;
    if (maxall > 0.0) std::frexp(maxall, &ye);
    p.fbits = f;
    p.ybits = ye;
    p.centre = centre;
    p.nV = nv;
    const int Kw = Kp / 32;
    e.qv.assign(Kp, 0);
    long long qmax2 = 0;
    for (int k : P) {
        const long long q = out[k] ? 0 : std::llround(std::ldexp((double)y[k] - centre, f));
        if (q > QMAX || q < -QMAX) return fail(c, EPI_ERR_RANGE, "fixed-point phenotype out of range");
        qmax2 = std::max(qmax2, q * q);
        e.qv[k] = (int32_t)q;
    }
    // q^2 limbs: the smallest shift that fits four limbs (15 when |q| reaches QMAX)
    int zb = 0;
    while (std::llround(std::ldexp((double)qmax2, -zb)) > ZMAX) zb++;
    p.zbits = zb;
    if (!arrays) return EPI_OK;
    e.w.assign((size_t)(NWP + 3 + NWC) * Kp, 0);
    e.yc.assign(Kp, 0.0f);
    e.yw.assign((size_t)2 * Kp, 0.0f);
    e.vb.assign(Kw, 0u);
    e.mp.assign(Kp, MissPhen{});
    long long qsum = 0;
    double sq = 0.0, ys = 0.0, y2 = 0.0;
    for (int k : P) {
        const long long q = e.qv[k];
        const long long z = std::llround(std::ldexp((double)(q * q), -zb));
        int8_t lq[3], lz[4];
        if (!split_limbs(q, 3, lq) || !split_limbs(z, 4, lz)) return fail(c, EPI_ERR_RANGE, "limb overflow");
        e.w[0 * (size_t)Kp + k] = 1;
        for (int t = 0; t < 3; t++) e.w[(1 + t) * (size_t)Kp + k] = lq[t];
        for (int t = 0; t < 4; t++) e.w[(4 + t) * (size_t)Kp + k] = lz[t];
        MissPhen &mk = e.mp[k];
        mk.v = 1;
        mk.q = (int32_t)q;
        mk.z = (int32_t)z;
        p.zall += (double)z;
        mk.qf = (float)q;
        mk.zf = (float)z;
        qsum += q;
        sq += (double)q * (double)q;
        const double dv = (double)y[k] - centre;
        const float ycf = (float)std::ldexp(dv, -ye);
        e.yc[k] = ycf;
        e.yw[k] = plain_weight(ycf, k);
        e.yw[Kp + k] = plain_weight(ycf * ycf, k);
        ys += (double)ycf;
        y2 += (double)ycf * (double)ycf;
        e.vb[k >> 5] |= 1u << (k & 31);
    }
    for (int nd : {1, 2}) encode_screen(P, Kp, nd, e);
    int8_t *cw = e.w.data() + (size_t)(NWP + 3) * Kp;
    for (int k : P) {
        const int v = e.mp[k].sv[1], lo = (int8_t)(v & 255);
        cw[k] = (int8_t)e.mp[k].sv[0];
        cw[Kp + k] = (int8_t)lo;
        cw[2 * (size_t)Kp + k] = (int8_t)((v - lo) / 256);
    }
    for (int t = 0; t < p.nout; t++) {
        const double u = std::ldexp((double)y[e.oidx[t]] - centre, f);
        e.ov.d[t] = u;
        e.ov.f[t] = (float)u;
        p.ouSum += u;
        p.ouSq += u * u;
    }
    p.qV = qsum;
    p.sqV = sq;
    p.ysV = ys;
    p.y2V = y2;
    return EPI_OK;
}

// Encode every phenotype on the host, then allocate and upload. On any
// failure the dataset is left without phenotypes (a scan then reports
// EPI_ERR_STATE), never with a partly built set.
int ds_set_phenotypes(epi_ctx *c, Dataset &d, const float *phen, int nphen, int nid, int flags)
{
    const bool nine_value = (flags & EPI_PHEN_NINE_IS_VALUE) != 0;
    if (!phen || nphen < 1 || nid < 2) return fail(c, EPI_ERR_ARG, "need phenotypes");
    if (nid > MAX_NID) return fail(c, EPI_ERR_RANGE, "nid %d above the supported %d", nid, MAX_NID);
    if (d.nid && nid != d.nid) return fail(c, EPI_ERR_ARG, "nid %d differs from genotypes' nid %d", nid, d.nid);
    drop_phenotypes(d);
    const int Kp = (nid + KPAD - 1) / KPAD * KPAD, Kw = Kp / 32;
    std::vector<PhenEnc> enc(nphen);
    for (int r = 0; r < nphen; r++) {
        int rc = encode_phen(c, phen + (size_t)r * nid, nid, Kp, nine_value, r, true, enc[r]);
        if (rc) return rc;
    }
    std::vector<PhenDev> ph(nphen);
    int rc = EPI_OK;
    for (int r = 0; r < nphen && rc == EPI_OK; r++) {
        PhenEnc &e = enc[r];
        PhenDev &p = ph[r];
        p = e.p;
        // one allocation and one copy: weights (with the screen's), mp, yc, yw, vbits (Kp is a multiple of 256), ov, oidx
        const size_t omp = e.w.size(), oyc = omp + (size_t)Kp * sizeof(MissPhen), oyw = oyc + (size_t)Kp * 4,
                     ovb = oyw + (size_t)Kp * 8, oov = ovb + (size_t)Kw * 4, oix = oov + sizeof(OutVals);
        std::vector<int8_t> blob(oix + sizeof(int32_t) * OUT_MAX, 0);
        memcpy(blob.data(), e.w.data(), e.w.size());
        memcpy(blob.data() + omp, e.mp.data(), (size_t)Kp * sizeof(MissPhen));
        memcpy(blob.data() + oyc, e.yc.data(), (size_t)Kp * 4);
        memcpy(blob.data() + oyw, e.yw.data(), (size_t)Kp * 8);
        memcpy(blob.data() + ovb, e.vb.data(), (size_t)Kw * 4);
        memcpy(blob.data() + oov, &e.ov, sizeof(OutVals));
        if (p.nout) memcpy(blob.data() + oix, e.oidx.data(), (size_t)p.nout * 4);
        if ((rc = dalloc(c, p.wts, blob.size()))) break;
        p.sw[0] = reinterpret_cast<uint32_t *>(p.wts + (size_t)NWP * Kp);
        p.sw[1] = p.sw[0] + Kp / 4;
        p.mp = reinterpret_cast<MissPhen *>(p.wts + omp);
        p.yc = reinterpret_cast<float *>(p.wts + oyc);
        p.yw = reinterpret_cast<float *>(p.wts + oyw);
        p.vbits = reinterpret_cast<uint32_t *>(p.wts + ovb);
        p.ov = reinterpret_cast<OutVals *>(p.wts + oov);
        p.oidx = reinterpret_cast<int32_t *>(p.wts + oix);
        hipError_t he = hipMemcpyAsync(p.wts, blob.data(), blob.size(), hipMemcpyHostToDevice, c->stream);
        if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
        if (he != hipSuccess) rc = fail(c, EPI_ERR_HIP, "phenotype upload failed: %s", hipGetErrorString(he));
    }
    if (rc) {
        for (auto &p : ph) free_phen(p);
        return rc;
    }
    if (!d.nid) {
        d.nid = nid;
        d.Kp = Kp;
        d.Kw = Kw;
    }
    d.ph.swap(ph);
    d.marg_ok = false;
    return EPI_OK;
}

int ds_set_chromosomes(epi_ctx *c, Dataset &d, const int32_t *chrstart, const int32_t *chrsize, int nchr)
{
    if (!chrstart || !chrsize || nchr < 1) return fail(c, EPI_ERR_ARG, "need chromosomes");
    if (!d.nsnp) return fail(c, EPI_ERR_STATE, "set genotypes before chromosomes");
    std::vector<int> snpchr(d.nsnp, -1);
    for (int i = 0; i < nchr; i++) {
        if (chrsize[i] < 0 || chrstart[i] < 0 || (long long)chrstart[i] + chrsize[i] > d.nsnp)
            return fail(c, EPI_ERR_ARG, "chromosome %d out of range", i);
        for (int s = chrstart[i]; s < chrstart[i] + chrsize[i]; s++) {
            if (snpchr[s] >= 0) return fail(c, EPI_ERR_ARG, "chromosomes %d and %d overlap", snpchr[s], i);
            snpchr[s] = i;
        }
    }
    d.chrstart.assign(chrstart, chrstart + nchr);
    d.chrsize.assign(chrsize, chrsize + nchr);
    d.snpchr.swap(snpchr);
    drop_sparse(d);  // its virtual SNP order follows the chromosomes
    return EPI_OK;
}

// Per-SNP marginals and outlier codes of every phenotype (they depend on both
// the genotypes and the phenotypes).
int ds_marginals(epi_ctx *c, Dataset &d)
{
    if (d.marg_ok) return EPI_OK;
    if (!d.mbits) return fail(c, EPI_ERR_STATE, "genotypes not set");
    if (d.ph.empty()) return fail(c, EPI_ERR_STATE, "phenotypes not set");
    for (auto &p : d.ph) {
        // one allocation: the screen's marginals, then the others
        const size_t per = sizeof(Marg) + sizeof(ScrMarg);
        p.marg = nullptr;
        int rc = dalloc(c, p.sm, (per * d.nsnp + sizeof(ScrMarg) - 1) / sizeof(ScrMarg));
        if (rc) return rc;
        p.marg = reinterpret_cast<Marg *>(p.sm + d.nsnp);
        hipLaunchKernelGGL(marginals_kernel, dim3((d.nsnp + 63) / 64), dim3(256), 0, c->stream,
                           (const uint32_t *)d.mbits, d.Kw, d.nsnp, (const uint32_t *)p.vbits, (const float *)p.yc,
                           (const int32_t *)d.cls, (const int8_t *)p.wts,
                           (const int8_t *)(p.wts + (size_t)(NWP + 3) * d.Kp), p.marg, p.sm);
        HIPCHK(c, hipGetLastError());
        if (p.nout) {
            if ((rc = dalloc(c, p.ocodes, (size_t)(p.nout + 15) / 16 * d.nsnp))) return rc;
            hipLaunchKernelGGL(outlier_codes_kernel, dim3((d.nsnp + 255) / 256), dim3(256), 0, c->stream,
                               (const uint32_t *)d.mbits, d.Kw, d.nsnp, (const int32_t *)p.oidx, p.nout, p.ocodes);
            HIPCHK(c, hipGetLastError());
        }
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    d.marg_ok = true;
    return EPI_OK;
}

// Virtual SNP order of the SPARSE tiles: chromosome i starts at a multiple of
// 64, so that the a- or b-range of every tile (which starts at its
// chromosome's start plus a multiple of the tile height) is one 64-SNP word,
// or half of one for 32-row tiles. Returns the number of words.
long long virtual_order(const Dataset &d, std::vector<int32_t> &vidx, std::vector<int32_t> *snp_of_v)
{
    vidx.assign(d.nsnp, 0);
    long long nv = 0;
    for (size_t i = 0; i < d.chrstart.size(); i++) {
        for (int t = 0; t < d.chrsize[i]; t++) vidx[d.chrstart[i] + t] = (int32_t)(nv + t);
        nv += (d.chrsize[i] + 63) / 64 * 64;
    }
    if (nv == 0) nv = 64;
    if (snp_of_v) {
        snp_of_v->assign(nv, -1);
        for (size_t i = 0; i < d.chrstart.size(); i++)
            for (int t = 0; t < d.chrsize[i]; t++) (*snp_of_v)[vidx[d.chrstart[i] + t]] = d.chrstart[i] + t;
    }
    return nv / 64;
}

// Device data of the SPARSE tiles for the current genotypes and chromosomes
// (the miss lists, the virtual SNP order and the transposed bitplanes), built
// when the genotypes or the chromosomes are set, for datasets with missing
// calls.
int ds_sparse(epi_ctx *c, Dataset &d)
{
    drop_sparse(d);
    if (!d.mbits || d.missc.empty() || d.missc[d.nsnp] == 0) return EPI_OK;
    std::vector<int32_t> vidx, sov;
    const long long nw = virtual_order(d, vidx, &sov);
    std::vector<long long> moff(d.nsnp + 1, 0);
    for (int s = 0; s < d.nsnp; s++) moff[s + 1] = moff[s] + d.miss[s];
    d.tstride = 4LL * d.nid;
    int32_t *dsov = nullptr;
    int rc;
    if ((rc = dalloc(c, d.moff, (size_t)d.nsnp + 1)) || (rc = dalloc(c, d.mlist, (size_t)std::max(1LL, moff[d.nsnp]))) ||
        (rc = dalloc(c, d.vidx, (size_t)d.nsnp)) || (rc = dalloc(c, d.tbits, (size_t)nw * d.tstride)) ||
        (rc = dalloc(c, dsov, sov.size()))) {
        dfree(dsov);
        drop_sparse(d);
        return rc;
    }
    hipError_t he = hipMemcpyAsync(d.moff, moff.data(), moff.size() * sizeof(long long), hipMemcpyHostToDevice,
                                   c->stream);
    if (he == hipSuccess)
        he = hipMemcpyAsync(d.vidx, vidx.data(), vidx.size() * sizeof(int32_t), hipMemcpyHostToDevice, c->stream);
    if (he == hipSuccess)
        he = hipMemcpyAsync(dsov, sov.data(), sov.size() * sizeof(int32_t), hipMemcpyHostToDevice, c->stream);
    if (he == hipSuccess) {
        hipLaunchKernelGGL(miss_list_kernel, dim3((d.nsnp + 255) / 256), dim3(256), 0, c->stream,
                           (const uint32_t *)d.mbits, d.Kw, d.nsnp, d.nid, (const long long *)d.moff, d.mlist);
        he = hipGetLastError();
    }
    if (he == hipSuccess) {
        hipLaunchKernelGGL(tbits_kernel, dim3((unsigned)nw, (d.nid + 31) / 32), dim3(64), 0, c->stream,
                           (const uint32_t *)d.mbits, d.Kw, d.nsnp, d.nid, (const int32_t *)dsov, (int)nw, d.tbits);
        he = hipGetLastError();
    }
    if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
    dfree(dsov);
    if (he != hipSuccess) {
        drop_sparse(d);
        return fail(c, EPI_ERR_HIP, "SPARSE tile data: %s", hipGetErrorString(he));
    }
    d.sp_ok = true;
    return EPI_OK;
}

// SPARSE tiles serve MFMA scans of datasets whose SPARSE data are built; the
// schedule can turn them off.
bool use_sparse(const Dataset &d, int form, const epi_schedule &sc)
{
    return form == EPI_FORM_MFMA && sc.dense_missing != 1 && d.sp_ok;
}

// MFMA scans of phenotype r need a phenotype the fixed point holds to 1e-5.
int check_mfma_phen(epi_ctx *c, const Dataset &d, int r)
{
    if (r >= 0 && r < (int)d.ph.size() && !d.ph[r].mfma_ok) return fail(c, EPI_ERR_RANGE, "%s", d.ph[r].mfma_why.c_str());
    return EPI_OK;
}

MfmaScan mfma_scan(const Dataset &d, int r, int tag)
{
    const PhenDev &p = d.ph[r];
    MfmaScan S;
    S.bits = d.mbits;
    S.sbits = d.sbits;
    S.wts = p.wts;
    S.marg = p.marg;
    S.nsnp = d.nsnp;
    S.Kp = d.Kp;
    S.Kl = (d.nid + KC - 1) / KC * KC;
    S.nV = p.nV;
    S.tag = tag;
    S.qV = p.qV;
    S.qVd = (double)p.qV;
    S.sqV = p.sqV;
    S.zunit = std::ldexp(1.0, p.zbits);
    S.ocodes = p.ocodes;
    S.ov = p.ov;
    S.nout = p.nout;
    S.ouSum = p.ouSum;
    S.ouSq = p.ouSq;
    S.tbits = d.tbits;
    S.vidx = d.vidx;
    S.moff = d.moff;
    S.mlist = d.mlist;
    S.mp = p.mp;
    S.tstride = d.tstride;
    S.rbits = d.bits;
    S.sw[0] = p.sw[0];
    S.sw[1] = p.sw[1];
    S.sm = p.sm;
    return S;
}

PlainScan plain_scan(const Dataset &d, int r, int tag)
{
    const PhenDev &p = d.ph[r];
    PlainScan S;
    S.bits = d.bits;
    S.yw = p.yw;
    S.vbits = p.vbits;
    S.marg = p.marg;
    S.nsnp = d.nsnp;
    S.Kw = d.Kw;
    S.nw = (d.nid + 31) / 32;
    S.nV = p.nV;
    S.tag = tag;
    S.ysV = p.ysV;
    S.y2V = p.y2V;
    return S;
}

// ------------------------------------------------------- no allocation --
// Scratch of epi_scan_noalloc: the hit counter in the first 256 bytes, then
// the tile list. Each device holds its own copy until the process ends. Host
// code reaches it only through the address hipGetSymbolAddress returns on
// that device (scratch_of), never through the array's name, which on the
// host is a stand-in and no device address.
constexpr size_t NOALLOC_BYTES = (size_t)16 << 20;
constexpr size_t NOALLOC_TILES = (NOALLOC_BYTES - 256) / sizeof(int4);
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

std::mutex scratch_mu;
std::vector<void *> scratch_ptr;  // per device ordinal

// This device's scratch address, looked up once per device (the device must be current).
int scratch_of(epi_ctx *c, void **out)
{
    std::lock_guard<std::mutex> g(scratch_mu);
    if ((int)scratch_ptr.size() <= c->device) scratch_ptr.resize(c->device + 1, nullptr);
    if (!scratch_ptr[c->device]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(c, EPI_ERR_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
        scratch_ptr[c->device] = ptr;
    }
    *out = scratch_ptr[c->device];
    return EPI_OK;
}

// Clears the hit counter with a kernel (no memset node in a captured stream).
__global__ void zero_counter(unsigned long long *n) { *n = 0ull; }

// Schedules. FAST tiles (no missing call in either SNP range) are
// fast_rows x 64. GENERAL tiles are fast_rows x 32 in the MFMA form (the
// same workgroup size as its FAST tiles, two waves per SIMD) and 16 x 64 in
// the plain form.
constexpr int TILE_B = 64;

int gen_rows(int form, const epi_schedule &s) { return form == EPI_FORM_MFMA ? s.fast_rows : 16; }
int gen_cols(int form, const epi_schedule &) { return form == EPI_FORM_MFMA ? 32 : 64; }

epi_schedule default_schedule(int form)
{
    epi_schedule s;
    memset(&s, 0, sizeof(s));
    // 32-row MFMA tiles keep two workgroups per CU (measured faster than 64
    // rows at N=4000 with missing calls and at N=8000 without)
    s.fast_rows = 32;
    s.super_a = 8;
    s.super_b = 4;
    s.queues = 8;
    s.order = 0;
    return s;
}

bool valid_schedule(int form, const epi_schedule &s)
{
    bool rows = form == EPI_FORM_MFMA ? (s.fast_rows == 64 || s.fast_rows == 32)
                                      : (s.fast_rows == 32 || s.fast_rows == 16);
    return rows && s.super_a >= 1 && s.super_a <= 64 && s.super_b >= 1 && s.super_b <= 64 &&
           (s.queues == 1 || s.queues == 8) && s.order >= 0 && s.order <= 2 &&
           (s.dense_missing >= 0 && s.dense_missing <= 2);
}

bool same_schedule(const epi_schedule &x, const epi_schedule &y)
{
    return x.fast_rows == y.fast_rows && x.super_a == y.super_a && x.super_b == y.super_b && x.queues == y.queues &&
           x.order == y.order && x.dense_missing == y.dense_missing;
}

void emit_tile(const Dataset &d, int a0, int a1, int b0, int b1, int grows, int gcols, bool sparse, bool sparse_all,
               TileLists &out)
{
    auto anymiss = [&](int s0, int s1) { return d.missc[s1] - d.missc[s0] > 0; };
    auto anyheavy = [&](int s0, int s1) { return d.heavyc[s1] - d.heavyc[s0] > 0; };
    if (a1 - 1 <= b0) return;  // no pair with a > b
    if (!anymiss(a0, a1) && !anymiss(b0, b1)) {
        out.fast.push_back(make_int4(a0, a1, b0, b1));
        return;
    }
    const long long nmiss = d.missum[a1] - d.missum[a0] + d.missum[b1] - d.missum[b0];
    if (sparse && !anyheavy(a0, a1) && !anyheavy(b0, b1) &&
        (sparse_all || nmiss * SPARSE_RATE <= (long long)(a1 - a0 + b1 - b0) * d.nid)) {
        out.sp.push_back(make_int4(a0, a1, b0, b1));
        return;
    }
    for (int x = a0; x < a1; x += grows) {
        int x1 = std::min(a1, x + grows);
        for (int y = b0; y < b1; y += gcols) {
            int y1 = std::min(b1, y + gcols);
            if (x1 - 1 <= y) continue;
            out.gen.push_back(make_int4(x, x1, y, y1));
        }
    }
}

// Pairs (a > b) of the chr x chr blocks [bb, be).
long long block_pairs(const Dataset &d, int bb, int be)
{
    long long n = 0;
    const int nchr = (int)d.chrstart.size();
    for (int i = 0; i < nchr; i++)
        for (int j = 0; j <= i; j++) {
            const int blk = i * (i + 1) / 2 + j;
            if (blk < bb || blk >= be) continue;
            // a in [A0, A1) meets b in [B0, min(B1, a))
            const long long A0 = d.chrstart[i], A1 = A0 + d.chrsize[i], B0 = d.chrstart[j], B1 = B0 + d.chrsize[j];
            const long long lo = std::max(A0, B0 + 1), mid = std::min(std::max(lo, B1), std::max(lo, A1));
            n += (mid - lo) * (lo - B0 + mid - 1 - B0) / 2;  // b up to a - 1
            if (A1 > mid) n += (A1 - mid) * std::max(0ll, B1 - B0);
        }
    return n;
}

// Where a piecewise tile build resumes: the next chr x chr block (index
// i(i+1)/2 + j) and, within it, the next super-tile row.
struct TileCursor {
    int blk = 0;
    int sa = 0;
};

// Tiles over the chr x chr blocks [cur.blk, blk_end). Within a block the
// tiles are emitted in super-tiles of super_a x super_b tiles so that
// neighbouring workgroups share SNP data in L2. The build stops after the
// super-tile row in which the list reaches max_tiles (a soft bound: one row
// of super-tiles is never split) and leaves cur at the next row; it returns
// true once the block range is exhausted. A block's pairs are counted with
// its first row.
bool build_tiles(const Dataset &d, int blk_end, int form, const epi_schedule &sc, size_t max_tiles, TileCursor &cur,
                 TileLists &out)
{
    const int TA = sc.fast_rows, TB = TILE_B, grows = gen_rows(form, sc), gcols = gen_cols(form, sc);
    const int nchr = (int)d.chrstart.size();
    const int SA = sc.super_a, SB = sc.super_b;
    const bool sparse = use_sparse(d, form, sc), sparse_all = sc.dense_missing == 2;
    for (int i = 0; i < nchr; i++) {
        for (int j = 0; j <= i; j++) {
            int blk = i * (i + 1) / 2 + j;
            if (blk < cur.blk) continue;
            if (blk >= blk_end) return true;
            cur.blk = blk;
            int A0 = d.chrstart[i], A1 = A0 + d.chrsize[i];
            int B0 = d.chrstart[j], B1 = B0 + d.chrsize[j];
            if (A1 <= A0 || B1 <= B0) {
                cur.sa = 0;
                continue;
            }
            if (cur.sa == 0) out.pairs += block_pairs(d, blk, blk + 1);
            int nta = (A1 - A0 + TA - 1) / TA, ntb = (B1 - B0 + TB - 1) / TB;
            for (int sa = cur.sa; sa < nta; sa += SA) {
                for (int sb = 0; sb < ntb; sb += SB)
                    for (int ta = sa; ta < std::min(nta, sa + SA); ta++)
                        for (int tb = sb; tb < std::min(ntb, sb + SB); tb++) {
                            int a0 = A0 + ta * TA, a1 = std::min(A1, a0 + TA);
                            int b0 = B0 + tb * TB, b1 = std::min(B1, b0 + TB);
                            emit_tile(d, a0, a1, b0, b1, grows, gcols, sparse, sparse_all, out);
                        }
                if (out.count() >= max_tiles && sa + SA < nta) {
                    cur.sa = sa + SA;
                    return false;
                }
            }
            cur.sa = 0;
            if (out.count() >= max_tiles) {
                cur.blk = blk + 1;
                return blk + 1 >= blk_end || blk + 1 >= nchr * (nchr + 1) / 2;
            }
        }
    }
    return true;
}

// The lists of one scan into dst, in device order (FAST, SPARSE, GENERAL).
int copy_tiles(epi_ctx *c, int4 *dst, const TileLists &tl)
{
    size_t o = 0;
    for (const std::vector<int4> *v : {&tl.fast, &tl.sp, &tl.gen}) {
        if (!v->empty())
            HIPCHK(c, hipMemcpyAsync(dst + o, v->data(), v->size() * sizeof(int4), hipMemcpyHostToDevice, c->stream));
        o += v->size();
    }
    return EPI_OK;
}

int upload_tiles(epi_ctx *c, const TileLists &tl, bool screen)
{
    c->tl_valid = false;
    // behind the tiles of a screened scan, room for the number and the mask of every block, of 64- or 32-row tiles
    const size_t nt = tl.count();
    size_t blocks = scr_blocks(64, 64, false) * (tl.fast.size() + tl.gen.size()) + scr_blocks(64, 64, true) * tl.sp.size();
    if (!screen) blocks = 0;
    const size_t need = nt + (2 * blocks * sizeof(uint32_t) + sizeof(int4) - 1) / sizeof(int4);
    static_assert(scr_blocks(64, 64, false) == scr_blocks(64, 32, true), "one count of blocks for FAST and GENERAL tiles");
    if (need > c->tiles_cap) {
        c->tiles_cap = 0;
        int rc = dalloc(c, c->tiles, need);
        if (rc) return rc;
        c->tiles_cap = need;
    }
    c->redo = screen ? reinterpret_cast<uint32_t *>(c->tiles + nt) : nullptr;
    c->redo_blocks = blocks;
    c->masks_set = false;
    return copy_tiles(c, c->tiles, tl);
}

HitSink make_sink(DevHit *hits, unsigned long long *nhits, long long cap, const epi_scan_params *p)
{
    HitSink hs;
    hs.hits = hits;
    hs.nhits = nhits;
    hs.cap = cap;
    hs.test = p->test;
    hs.t1 = p->t1;
    hs.t2 = p->t2;
    hs.t1s = p->t1 * 0.98f;
    hs.t2s = p->t2 * 0.98f;
    hs.tag = p->phen;
    hs.safe = p->safe ? 1 : 0;
    return hs;
}

int check_common(epi_ctx *c, const epi_scan_params *p)
{
    if (!p) return fail(c, EPI_ERR_ARG, "null params");
    if (p->test != 'f' && p->test != 'i') return fail(c, EPI_ERR_ARG, "test must be 'f' or 'i'");
    if (p->form != EPI_FORM_PLAIN && p->form != EPI_FORM_MFMA) return fail(c, EPI_ERR_ARG, "unknown form");
    if (!(p->t1 == p->t1) || !(p->t2 == p->t2)) return fail(c, EPI_ERR_ARG, "threshold is NaN");
    return EPI_OK;
}

int check_params(epi_ctx *c, const epi_scan_params *p)
{
    int rc = check_common(c, p);
    if (rc) return rc;
    if (!c->d.mbits) return fail(c, EPI_ERR_STATE, "genotypes not set");
    if (c->d.ph.empty()) return fail(c, EPI_ERR_STATE, "phenotypes not set");
    if (p->phen < 0 || p->phen >= (int)c->d.ph.size()) return fail(c, EPI_ERR_ARG, "phenotype index out of range");
    if (c->d.chrstart.empty()) return fail(c, EPI_ERR_STATE, "chromosomes not set");
    if (p->form == EPI_FORM_MFMA) return check_mfma_phen(c, c->d, p->phen);
    return EPI_OK;
}

// A launch covers at most 2^31 work-items (the runtime counts the global size in 32 bits; beyond 2^32 it
// would launch only the wrapped remainder), so a long tile list goes out as several launches, each over its
// own slice of the list and a whole number of 256-workgroup groups (the XCD mapping of xcd_tile).
#define LAUNCH_TILES(KERNEL, THREADS, ARGS, FIRST, N)                                                   \
    do {                                                                                                 \
        const int chunk_ = (int)((1u << 31) / (unsigned)(THREADS)) & ~255;                              \
        for (int t0_ = 0; t0_ < (N); t0_ += chunk_) {                                                    \
            (ARGS).tiles = (FIRST) + t0_;                                                                \
            (ARGS).ntiles = std::min(chunk_, (N) - t0_);                                                 \
            hipLaunchKernelGGL(KERNEL, dim3((ARGS).ntiles), dim3(THREADS), 0, c->stream, (ARGS));        \
            HIPCHK(c, hipGetLastError());                                                                \
            c->last_launches++;                                                                          \
        }                                                                                                \
    } while (0)

// Device buffers of a scan's pair kernels: the tile list, the hit records and the hit counter, and
// the screen's sink (no screen without it).
struct ScanBufs {
    int4 *tiles;
    DevHit *hits;
    unsigned long long *nhits;
    long long cap;
    CandSink cs;
    unsigned long long *emptied;
};

ScanBufs ctx_bufs(const epi_ctx *c)
{
    return {c->tiles, c->hits, &c->count->nhits, c->cap, {c->cand, c->count->screen, CAND_CAP, c->redo, c->redo + c->redo_blocks}, &c->count->emptied};
}

// Lanes per candidate of resolve_kernel for a cohort of Kl individuals (one 32-individual word each).
int resolve_lanes(int Kl)
{
    int g = 4;
    while (g < 64 && g * 32 < Kl) g *= 2;
    return g;
}

// Upper tail of chi-square with 2 h degrees of freedom.
double chi2_tail(double x, int h)
{
    double t = 1.0, sum = 1.0;
    for (int j = 1; j < h; j++) sum += t *= 0.5 * x / j;
    return std::exp(-0.5 * x) * sum;
}

// The screen's cut for a phenotype and the scan's thresholds; false where the
// exact tiles are the better path: thresholds so low, or a cohort so large for
// the coarse phenotype's residue, that more than SCR_RATE2 of the pairs of
// unrelated SNPs would be candidates. One digit (two thirds of the MFMAs) where SCR_RATE1 holds with it: its
// larger residue sends more pairs to the second stage and to the resolve kernel (M = 20000, normal phenotype, no
// missing calls: N = 1500, test i, rate 8e-5: 1.35 ms against 1.57 ms with two digits; N = 3000, test f, 4e-4:
// 0.87-0.96 of two digits by phenotype, but with 1 % missing calls 0.91-1.03; N = 3000, test i, 7e-4: 3.02 against 2.64).
constexpr double SCR_RATE1 = 2.5e-4, SCR_RATE2 = 2e-3;
// Pairs times individuals below which the screen's further launches (measured with two) cost more than its
// kernel saves (N = 1000, M = 1000: 20.5 us either way; N = 300, M = 2000: 25.9 us exact, 18.0 us screened).
constexpr double SCR_MIN_WORK = 5e8;

bool screen_cut(const PhenDev &p, const epi_scan_params *q, ScreenCut &C)
{
    const HitSink hs = make_sink(nullptr, nullptr, 0, q);
    if (p.nout || p.nV < 32 || !(hs.t1s > 0.0f)) return false;
    const bool inter = q->test != 'f';
    if (inter && !(hs.t2s > 0.0f)) return false;
    if (!std::isfinite(hs.t1s) || (inter && !std::isfinite(hs.t2s))) return false;
    const double N = p.nV, qV = (double)p.qV, sst = p.sqV - qV * qV / N, sig2 = sst / (N - 1.0);
    if (!(sst > 0.0)) return false;
    // F > t1 is SSB > k1 SST, and F2 > t2 takes SSB >= SSI > k2 SST; n complete cases
    auto k1 = [&](int nfac, double n) {
        const double k = (double)hs.t1s * (nfac - 1);
        return k / (n - nfac + k);
    };
    auto k2 = [&](int nfac, double n) {
        const double k = 4.0 * (double)hs.t2s;
        return k / (n - nfac + k);
    };
    auto kap = [&](int nfac, double n) { return inter ? std::min(k1(nfac, n), k2(nfac, n)) : k1(nfac, n); };
    int nd = 0;
    double rate = 0.0;
    for (int i = 1; i <= 2 && !nd; i++) {
        const ScreenEnc &E = p.scr[i - 1];
        if (!(E.delta > 0.0)) continue;
        auto tail = [&](double k, int h) { return chi2_tail(std::pow(std::max(0.0, std::sqrt(k * sst) - E.eps), 2) / sig2, h); };
        rate = tail(k1(9, N), 4);
        if (inter) rate += tail(k2(9, N), 2);
        if (rate <= (i == 1 ? SCR_RATE1 : SCR_RATE2)) nd = i;
    }
    if (!nd) return false;
    const ScreenEnc &E = p.scr[nd - 1];
    const double unit = 64.0 * E.delta * E.delta;  // q^2 units per unit of the kernels' sums of squares
    memset(&C, 0, sizeof(C));
    const double T = E.vsum / 64.0, T2N = T * T / (N / 64.0);
    // level 0 of FAST tiles: a lower bound on sum s^2 / n = SSB(v) + T^2 / N, linear in the occupied cells
    auto level0 = [&](int nfac) {
        return (std::pow(std::max(0.0, std::sqrt(kap(nfac, N) * sst) - E.eps), 2) / unit + T2N) * (1.0 - 1e-5);
    };
    const int least = inter && !q->safe ? 7 : 2;  // occupied cells of a hit
    const double thr9 = level0(9);
    double slope = 0.0;
    for (int k = least; k < 9; k++) slope = std::max(slope, (thr9 - level0(k)) / (9 - k));
    slope *= 1.0 + 1e-5;
    C.thr0 = (float)((thr9 - 9.0 * slope) - 1e-5 * std::fabs(thr9 - 9.0 * slope));
    C.slope2 = (float)(0.5 * slope);
    C.eps = (float)(E.eps / (8.0 * E.delta) * (1.0 + 1e-6));
    C.sst = (float)(sst / unit * (1.0 - 1e-6));
    C.nv = (float)N;
    C.N = (float)(N / 64.0);
    C.t1s = hs.t1s;
    C.t2s = hs.t2s;
    C.test = q->test;
    C.safe = hs.safe;
    C.nd = nd;
    C.rate = (float)rate;
    // GENERAL tiles: the pair's complete cases N' <= N and their SST vary. k / (N' - nfac + k) is smallest at
    // N' = N; the linear form of (sqrt(k SST) - eps)^2 >= k SST - 2 eps sqrt(k SST) takes the largest
    // k SST at N' >= N / 2 (pairs with fewer skip level 0).
    const double k9 = kap(9, N) * (1.0 - 1e-5);
    double ks = 0.0;
    for (int k = least; k < 9; k++) ks = std::max(ks, (k9 - kap(k, N) * (1.0 - 1e-5)) / (9 - k));
    ks *= 1.0 + 1e-5;
    C.kap0 = (float)((k9 - 9.0 * ks) - 1e-5 * std::fabs(k9 - 9.0 * ks));
    C.kslope2 = (float)(0.5 * ks);
    C.kroot = (float)(2.0 * E.eps * std::sqrt(kap(9, std::max(0.5 * N, 16.0)) * p.sqV) / unit * (1.0 + 1e-5));
    C.vs = (float)(E.vsum / 64.0);
    C.zunit = (float)(std::ldexp(1.0, p.zbits) / unit * (1.0 - 1e-6));
    C.zall = (float)(p.zall * (1.0 + 1e-6));
    C.c0 = (float)(E.offset / E.delta);
    return true;
}

// The screen's 32-bit offsets reach two bitplanes (planes_fit), and
// GENERAL tiles bound SST well up to an eighth of the calls missing.
bool screen_fits(const Dataset &d)
{
    return planes_fit(d) && d.missum[d.nsnp] <= (long long)d.nsnp * d.nid / 8;
}

// One kind of tile through the screen. tiles: the kind's list on the device.
struct ScreenKind {
    const int4 *tiles;
    int n;
    uint32_t *count;   // candidates and blocks of this kind
    uint32_t *redo, *mask;
    unsigned long long *emptied;
};

// Launches of the bound and the resolve kernel, a list of candidates at a time; or, once the host has their counters, of the redo of K's blocks.
template <bool GEN, int TA, int TB>
int launch_screen(epi_ctx *c, ScreenArgs &G, const HitSink &hs, const ScreenKind &K, uint32_t redo)
{
    if (redo) {
        const RedoArgs D = {G.S, nullptr, hs, K.tiles, K.count, K.redo, K.mask};
        hipLaunchKernelGGL((redo_kernel<TA, TB, GEN, false>), dim3(std::min(redo, 1u << 22)), dim3(256), 0, c->stream, D);
        HIPCHK(c, hipGetLastError());
        c->last_launches++;
        return EPI_OK;
    }
    G.cs.count = K.count;
    G.cs.redo = K.redo;
    G.cs.mask = K.mask;
    G.halves = GEN ? TB / 32 : 1;
    const ResolveArgs R = {G.S, nullptr, hs, G.cs.cand, K.count, G.cs.cap, resolve_lanes(G.S.Kl)};
    const int most = scr_chunk(G.cut.rate, TA, TB, scr_threads<TA>() * G.halves);
    for (int t0 = 0; t0 < K.n;) {
        const int chunk = std::min(most, K.n - t0);
        const dim3 grid(chunk * G.halves), block(scr_threads<TA>());
        G.tiles = K.tiles + t0;
        G.ntiles = chunk;
        G.tile0 = t0;
        if constexpr (GEN) {
            constexpr bool NC = TA == 64;
            const bool nocall = NC && scr_nocall(G.S.Kl);
            if (G.cut.nd == 1) {
                if (nocall) hipLaunchKernelGGL((screen_gen_kernel<TA, 1, NC>), grid, block, 0, c->stream, G);
                else hipLaunchKernelGGL((screen_gen_kernel<TA, 1, false>), grid, block, 0, c->stream, G);
            } else {
                if (nocall) hipLaunchKernelGGL((screen_gen_kernel<TA, 2, NC>), grid, block, 0, c->stream, G);
                else hipLaunchKernelGGL((screen_gen_kernel<TA, 2, false>), grid, block, 0, c->stream, G);
            }
        } else {
            if (G.cut.nd == 1) hipLaunchKernelGGL((screen_fast_kernel<TA, 1>), grid, block, 0, c->stream, G);
            else hipLaunchKernelGGL((screen_fast_kernel<TA, 2>), grid, block, 0, c->stream, G);
        }
        HIPCHK(c, hipGetLastError());
        hipLaunchKernelGGL((resolve_kernel<GEN, false>), dim3(4 * c->ncu), dim3(256), 0, c->stream, R);
        HIPCHK(c, hipGetLastError());
        c->last_launches += 2;
        t0 += chunk;
        if (t0 == K.n) break;
        hipLaunchKernelGGL(empty_list, dim3(1), dim3(1), 0, c->stream, K.count, G.cs.cap, K.emptied);
        HIPCHK(c, hipGetLastError());
        c->last_launches++;
    }
    return EPI_OK;
}

// Tile height of a screened scan. The K loop of a small cohort's tile is short, and workgroups of two waves overlap
// their starts and ends better (kernel time of 64 rows over 32: N = 500 to 1500 1.02 to 1.04 without missing calls and
// 1.01 to 1.03 with 1 or 2 %, N = 2000 1.02 and 0.98, N = 3000 0.99 and 0.95, N = 20000 0.99 and 0.97); the list of 64-row tiles is half as
// long, which a first scan pays for on the host.
int screen_rows(int nid) { return nid >= 2000 ? 64 : 32; }

// Whether the scan of phenotype p.phen over `pairs` pairs goes through the screen, and its cut.
bool screened(const Dataset &d, const epi_scan_params *p, long long pairs, ScreenCut &C)
{
    const double unit = d.missum[d.nsnp] ? 2.5 : 1.0;  // of the exact tiles' cost
    return p->form == EPI_FORM_MFMA && unit * (double)pairs * d.nid >= SCR_MIN_WORK && screen_fits(d) &&
           screen_cut(d.ph[p->phen], p, C);
}

// Launch the pair kernels of one scan over the uploaded tile lists (fast tiles first).
// counts: the screen's counters of an earlier call, whose blocks are to be redone (nothing else is launched).
template <bool DUMP>
int launch_pairs(epi_ctx *c, const epi_scan_params *p, const epi_schedule &sc, const TileLists &tl,
                 const DumpSink &ds, const ScanBufs &B, const ScreenCut *cut = nullptr, const uint32_t *counts = nullptr)
{
    const Dataset &d = c->d;
    if (tl.count() > (size_t)INT32_MAX)
        return fail(c, EPI_ERR_RANGE, "a super-tile row of this scan exceeds 2^31 tiles");
    const int nf = (int)tl.fast.size(), ns = (int)tl.sp.size(), ng = (int)tl.gen.size();
    if (tl.count() > SCR_TILES) cut = nullptr;  // one row of super-tiles beyond what the screen can number
    c->last_launches = 0;
    if (!counts) {
        c->last_tiles[0] += nf;
        c->last_tiles[1] += ns;
        c->last_tiles[2] += ng;
    }
    const HitSink hs = make_sink(B.hits, B.nhits, B.cap, p);
    if (p->form == EPI_FORM_MFMA) {
        MfmaArgs A;
        A.S = mfma_scan(d, p->phen, p->phen);
        A.hs = hs;
        A.ds = ds;
        if (ns && !d.sp_ok) return fail(c, EPI_ERR_STATE, "SPARSE tile data not built");
        // Every kind of tile goes through the screen with a cut (SPARSE tiles that the schedule asks for do not).
        const bool sf = cut && nf, ss = cut && ns && sc.dense_missing != 2, sg = cut && ng;
        if (sf || ss || sg) {
            ScreenArgs G;
            G.S = A.S;
            G.cut = *cut;
            G.cs = B.cs;
            const size_t of = scr_blocks(64, 64, false) * (size_t)nf, os = of + scr_blocks(64, 64, true) * (size_t)ns;
            const ScreenKind kf = {B.tiles, nf, B.cs.count, B.cs.redo, B.cs.mask, B.emptied},
                             ks = {B.tiles + nf, ns, B.cs.count + 2, B.cs.redo + of, B.cs.mask + of, B.emptied},
                             kg = {B.tiles + nf + ns, ng, B.cs.count + 4, B.cs.redo + os, B.cs.mask + os, B.emptied};
            const bool again = counts != nullptr;
            const bool lf = sf && (!again || counts[1]), ls = ss && (!again || counts[3]), lg = sg && (!again || counts[5]);
            const uint32_t rf = again ? counts[1] : 0u, rs = again ? counts[3] : 0u, rg = again ? counts[5] : 0u;
            int rc = EPI_OK;
            if (sc.fast_rows == 64) {
                if (lf) rc = launch_screen<false, 64, 64>(c, G, hs, kf, rf);
                if (ls && !rc) rc = launch_screen<true, 64, 64>(c, G, hs, ks, rs);
                if (lg && !rc) rc = launch_screen<true, 64, 32>(c, G, hs, kg, rg);
            } else {
                if (lf) rc = launch_screen<false, 32, 64>(c, G, hs, kf, rf);
                if (ls && !rc) rc = launch_screen<true, 32, 64>(c, G, hs, ks, rs);
                if (lg && !rc) rc = launch_screen<true, 32, 32>(c, G, hs, kg, rg);
            }
            if (rc || again) return rc;
        }
        const int xf = sf ? 0 : nf, xs = ss ? 0 : ns, xg = sg ? 0 : ng;  // tiles left to the exact kernels
        if (sc.fast_rows == 64) {
            LAUNCH_TILES((mfma_fast_kernel<64, DUMP>), fast_threads<64>(), A, B.tiles, xf);
            LAUNCH_TILES((mfma_sparse_kernel<64, DUMP>), sparse_threads<64>(), A, B.tiles + nf, xs);
            LAUNCH_TILES((mfma_general_kernel<64, DUMP>), general_threads<64>(), A, B.tiles + nf + ns, xg);
        } else {
            LAUNCH_TILES((mfma_fast_kernel<32, DUMP>), fast_threads<32>(), A, B.tiles, xf);
            LAUNCH_TILES((mfma_sparse_kernel<32, DUMP>), sparse_threads<32>(), A, B.tiles + nf, xs);
            LAUNCH_TILES((mfma_general_kernel<32, DUMP>), general_threads<32>(), A, B.tiles + nf + ns, xg);
        }
    } else {
        PlainArgs P;
        P.S = plain_scan(d, p->phen, p->phen);
        P.hs = hs;
        P.ds = ds;
        if (sc.fast_rows == 32)
            LAUNCH_TILES((plain_kernel<512, true, DUMP>), 512, P, B.tiles, nf);
        else
            LAUNCH_TILES((plain_kernel<256, true, DUMP>), 256, P, B.tiles, nf);
        LAUNCH_TILES((plain_kernel<256, false, DUMP>), 256, P, B.tiles + nf + ns, ng);
    }
    return EPI_OK;
}

// Order of the hits by (block, snp1, snp2): sorted[t] indexes h. A hit's key packs the three into 64 bits
// wherever they fit, and long lists go through a radix sort of eleven bits a pass (67,000 hits: 0.5 ms; 4.6 ms by
// comparisons that look the records up).
void sort_hits(const Dataset &d, const DevHit *h, const std::vector<int> &idx, std::vector<std::pair<uint64_t, int>> &sorted)
{
    auto bits = [](long long n) {
        int b = 0;
        while (n > 1ll << b) b++;
        return b;
    };
    const long long nchr = (long long)d.chrstart.size(), nblk = nchr * (nchr + 1) / 2;
    const int ns = bits(d.nsnp), total = bits(nblk) + 2 * ns;
    auto blk_of = [&](const DevHit &x) {
        const uint64_t i = d.snpchr[x.snp1], j = d.snpchr[x.snp2];
        return i * (i + 1) / 2 + j;
    };
    const size_t n = idx.size();
    sorted.resize(n);
    for (size_t t = 0; t < n; t++) {
        const DevHit &x = h[idx[t]];
        // (snp1, snp2) take at most 62 bits; the block is left to the comparison where all three do not fit
        sorted[t] = {(total <= 64 ? blk_of(x) << (2 * ns) : 0) | (uint64_t)x.snp1 << ns | (uint64_t)x.snp2, idx[t]};
    }
    if (total > 64) {
        std::sort(sorted.begin(), sorted.end(), [&](const auto &p, const auto &q) {
            const uint64_t bp = blk_of(h[p.second]), bq = blk_of(h[q.second]);
            return bp != bq ? bp < bq : p.first < q.first;
        });
    } else if (n < 512) {
        std::sort(sorted.begin(), sorted.end());
    } else {
        std::vector<std::pair<uint64_t, int>> other(n);
        for (int sh = 0; sh < total; sh += 11) {
            size_t at[2048] = {0}, sum = 0;
            for (const auto &x : sorted) at[x.first >> sh & 2047]++;
            for (size_t &a : at) {
                const size_t k = a;
                a = sum;
                sum += k;
            }
            for (const auto &x : sorted) other[at[x.first >> sh & 2047]++] = x;
            sorted.swap(other);
        }
    }
}

// Hits of one scan sorted by (block, snp1, snp2) and written out.
void emit_hits(const Dataset &d, const DevHit *h, const std::vector<int> &idx, epi_hit *hits, double *F64, double *F2_64,
               int32_t *block, long long cap, long long *n)
{
    std::vector<std::pair<uint64_t, int>> sorted;
    sort_hits(d, h, idx, sorted);
    const long long m = std::min<long long>((long long)sorted.size(), cap);
    for (long long t = 0; t < m; t++) {
        const DevHit &x = h[sorted[t].second];
        if (hits) {
            hits[t].snp1 = x.snp1;
            hits[t].snp2 = x.snp2;
            hits[t].df1 = x.df1;
            hits[t].df2 = x.df2;
            hits[t].F = (float)x.F;
            hits[t].F2 = (float)x.F2;
        }
        if (F64) F64[t] = x.F;
        if (F2_64) F2_64[t] = x.F2;
        if (block) {
            const int i = d.snpchr[x.snp1], j = d.snpchr[x.snp2];
            block[t] = i * (i + 1) / 2 + j;
        }
    }
    if (n) *n = m;
}

// ------------------------------------------------------------------ batch --

// Work items of every scan and the queue boundaries of the schedule.
// Per dataset the items are in locality order: tile-major (super-tiles),
// phenotype-minor, one list per tile kind. order 1 runs the GENERAL and
// SPARSE lists before the FAST one, order 2 takes datasets by decreasing Kp,
// so that the longest items do not end up in the tail. With 8 queues the list
// is cut into NQ contiguous pieces of equal estimated cost, one per XCD;
// with 1 queue every workgroup pulls from one shared queue.
// The scans of `scr` have lists of their own, with tiles of scr_rows.
constexpr size_t batch_blocks(int kind) { return scr_blocks(64, kind == 1 ? 32 : 64, kind != 0); }

int build_batch_work(epi_batch *b, int form, const epi_schedule &sched, const std::vector<char> &scr, int scr_rows)
{
    epi_ctx *c = b->ctx;
    const int nd = (int)b->data.size();
    std::vector<std::vector<int4>> wk[NLIST];
    std::vector<std::vector<double>> ct[NLIST];
    for (int l = 0; l < NLIST; l++) {
        wk[l].resize(nd);
        ct[l].resize(nd);
    }
    b->pairs = 0;
    // estimated cost per pair and individual, by kind
    const double unit[NKIND] = {form == EPI_FORM_MFMA ? 16.0 : 4.0, form == EPI_FORM_MFMA ? 40.0 : 10.0, 22.0};
    for (int i = 0; i < 2 * nd; i++) {
        const int di = i / 2, g = i % 2;
        const Dataset &d = *b->data[di];
        std::vector<int> sc;
        for (int s = 0; s < (int)b->scans.size(); s++)
            if (b->scans[s].first == di && !scr[s] == (g == 1)) sc.push_back(s);
        if (sc.empty()) continue;
        TileLists tl;
        TileCursor all;
        epi_schedule sg = sched;
        if (!g) sg.fast_rows = scr_rows;
        build_tiles(d, 1 << 30, form, sg, SIZE_MAX, all, tl);
        b->pairs += tl.pairs * (long long)sc.size();
        for (int kind = 0; kind < NKIND; kind++) {
            const std::vector<int4> &v = kind == 0 ? tl.fast : kind == 1 ? tl.gen : tl.sp;
            for (const int4 &t : v) {
                int ext = (t.y - t.x) | ((t.w - t.z) << 8) | (kind << 16);
                double cst = (double)(t.y - t.x) * (t.w - t.z) * d.Kp * unit[kind] + 5e4;
                for (int s : sc) {
                    wk[NKIND * g + kind][di].push_back(make_int4(t.x, t.z, ext, s));
                    ct[NKIND * g + kind][di].push_back(cst);
                }
            }
        }
    }
    std::vector<int> dorder(nd);
    for (int i = 0; i < nd; i++) dorder[i] = i;
    if (sched.order == 2)
        std::stable_sort(dorder.begin(), dorder.end(),
                         [&](int x, int y) { return b->data[x]->Kp > b->data[y]->Kp; });
    // One list per tile kind, each run by its own
    // kernel so that a kernel holds the registers of one tile kind only; within a list the datasets
    // follow the schedule's order. Each list is cut into its own queues.
    std::vector<int4> work;
    std::vector<int> qbegin(NLIST * NQ), qend(NLIST * NQ);
    for (int l = 0; l < NLIST; l++) {
        const int base = (int)work.size();
        std::vector<double> cost;
        if (l < NKIND) b->segs[l].clear();
        for (int di : dorder) {
            if (l < NKIND && !wk[l][di].empty()) b->segs[l].push_back({di, (long long)wk[l][di].size()});
            work.insert(work.end(), wk[l][di].begin(), wk[l][di].end());
            cost.insert(cost.end(), ct[l][di].begin(), ct[l][di].end());
        }
        static_assert(SCR_TILES > INT32_MAX / 2, "the screen numbers the blocks of any list");
        if (work.size() > (size_t)INT32_MAX / 2) return fail(c, EPI_ERR_RANGE, "batch has too many tiles");
        const int n = (int)work.size();
        b->nlist[l] = n - base;
        int *qb = qbegin.data() + l * NQ, *qe = qend.data() + l * NQ;
        for (int q = 0; q < NQ; q++) qb[q] = qe[q] = n;
        qb[0] = base;
        if (sched.queues == 1) {
            qe[0] = n;
        } else {
            double total = 0.0;
            for (double x : cost) total += x;
            double acc = 0.0;
            int q = 0;
            for (int i = base; i < n && q < NQ - 1; i++) {
                acc += cost[i - base];
                if (acc >= total * (q + 1) / NQ) {
                    qe[q] = i + 1;
                    qb[++q] = i + 1;
                }
            }
        }
    }
    b->nwork = (long long)work.size();
    int rc;
    // behind the items, room for the number and the mask of every block of the screen's tiles, of 64 or 32 rows
    size_t blocks = 0;
    for (int kind = 0; kind < NKIND; kind++) blocks += batch_blocks(kind) * (size_t)b->nlist[kind];
    const size_t room = work.size() + (2 * blocks * sizeof(uint32_t) + sizeof(int4) - 1) / sizeof(int4);
    if (room > b->work_cap) {
        b->work_cap = 0;
        if ((rc = dalloc(c, b->d_work, room))) return rc;
        b->work_cap = room;
    }
    b->redo = reinterpret_cast<uint32_t *>(b->d_work + work.size());
    b->mask = b->redo + blocks;
    HIPCHK(c, hipMemsetAsync(b->mask, 0, blocks * sizeof(uint32_t), c->stream));
    if (!work.empty())
        HIPCHK(c, hipMemcpyAsync(b->d_work, work.data(), work.size() * sizeof(int4), hipMemcpyHostToDevice,
                                 c->stream));
    HIPCHK(c, hipMemcpyAsync(b->d_qbegin, qbegin.data(), NLIST * NQ * sizeof(int), hipMemcpyHostToDevice,
                             c->stream));
    HIPCHK(c, hipMemcpyAsync(b->d_qend, qend.data(), NLIST * NQ * sizeof(int), hipMemcpyHostToDevice, c->stream));
    // scan descriptors
    size_t ns = b->scans.size();
    if (ns > b->scan_cap) {
        if ((rc = dalloc(c, b->d_mscan, ns)) || (rc = dalloc(c, b->d_pscan, ns)) || (rc = dalloc(c, b->d_cut, ns))) return rc;
        b->scan_cap = ns;
    }
    std::vector<MfmaScan> ms(ns);
    std::vector<PlainScan> ps(ns);
    for (size_t s = 0; s < ns; s++) {
        const Dataset &d = *b->data[b->scans[s].first];
        ms[s] = mfma_scan(d, b->scans[s].second, (int)s);
        ps[s] = plain_scan(d, b->scans[s].second, (int)s);
    }
    HIPCHK(c, hipMemcpyAsync(b->d_mscan, ms.data(), ns * sizeof(MfmaScan), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(b->d_pscan, ps.data(), ns * sizeof(PlainScan), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    b->work_form = form;
    b->work_sched = sched;
    b->work_scr = scr;
    b->scr_rows = scr_rows;
    b->dirty = false;
    return EPI_OK;
}

long long candidates(const Counters &n)
{
    long long c = (long long)n.emptied;
    for (int k = 0; k < NKIND; k++) c += std::min(n.screen[2 * k], CAND_CAP);
    return c;
}

long long redone(const Counters &n) { return (long long)n.screen[1] + n.screen[3] + n.screen[5]; }

bool same_key(const epi_scan_params &x, const epi_scan_params &y)
{
    return x.test == y.test && x.form == y.form && x.t1 == y.t1 && x.t2 == y.t2 && (x.safe != 0) == (y.safe != 0);
}

void drop_graph(epi_batch *b)
{
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    b->gvalid = false;
}

// Threads per workgroup of batch_kernel(form, sc, kind).
int batch_threads_of(int form, const epi_schedule &sc, int kind)
{
    if (form != EPI_FORM_MFMA) return kind ? 256 : 16 * sc.fast_rows;
    if (sc.fast_rows == 64)
        return kind == 2 ? batch_threads<64, 2>() : kind ? batch_threads<64, 1>() : batch_threads<64, 0>();
    return kind == 2 ? batch_threads<32, 2>() : kind ? batch_threads<32, 1>() : batch_threads<32, 0>();
}

const void *batch_kernel(int form, const epi_schedule &sc, int kind)
{
    if (form == EPI_FORM_MFMA) {
        if (sc.fast_rows == 64)
            return kind == 2 ? (const void *)mfma_batch_kernel<64, 2>
                   : kind    ? (const void *)mfma_batch_kernel<64, 1>
                             : (const void *)mfma_batch_kernel<64, 0>;
        return kind == 2 ? (const void *)mfma_batch_kernel<32, 2>
               : kind    ? (const void *)mfma_batch_kernel<32, 1>
                         : (const void *)mfma_batch_kernel<32, 0>;
    }
    // the plain form has no SPARSE tiles
    if (sc.fast_rows == 32)
        return kind ? (const void *)plain_batch_kernel<256, 1> : (const void *)plain_batch_kernel<512, 0>;
    return kind ? (const void *)plain_batch_kernel<256, 1> : (const void *)plain_batch_kernel<256, 0>;
}

// Whether a batch's screened tiles with missing calls contract those: one answer for the list, that of most of its work.
bool batch_nocall(const epi_batch *b)
{
    double large = 0.0, all = 0.0;
    for (size_t s = 0; s < b->scans.size(); s++) {
        const Dataset &d = *b->data[b->scans[s].first];
        if (!b->work_scr[s] || !d.missum[d.nsnp]) continue;
        const double w = (double)d.nsnp * d.nsnp * d.nid;
        all += w;
        if (scr_nocall((d.nid + KC - 1) / KC * KC)) large += w;
    }
    return 2.0 * large > all;
}

const void *screen_batch_fn(const epi_schedule &sc, int kind, bool nocall)
{
    if (sc.fast_rows == 64) {
        if (kind == 2) return nocall ? (const void *)screen_batch_kernel<64, 2, true> : (const void *)screen_batch_kernel<64, 2>;
        if (kind) return nocall ? (const void *)screen_batch_kernel<64, 1, true> : (const void *)screen_batch_kernel<64, 1>;
        return (const void *)screen_batch_kernel<64, 0>;
    }
    return kind == 2 ? (const void *)screen_batch_kernel<32, 2>
           : kind    ? (const void *)screen_batch_kernel<32, 1>
                     : (const void *)screen_batch_kernel<32, 0>;
}

const void *redo_batch_fn(const epi_schedule &sc, int kind)
{
    if (sc.fast_rows == 64)
        return kind == 2 ? (const void *)redo_kernel<64, 64, true, true>
               : kind    ? (const void *)redo_kernel<64, 32, true, true>
                         : (const void *)redo_kernel<64, 64, false, true>;
    return kind == 2 ? (const void *)redo_kernel<32, 64, true, true>
           : kind    ? (const void *)redo_kernel<32, 32, true, true>
                     : (const void *)redo_kernel<32, 64, false, true>;
}

// The scans' cuts and which of them go through the screen (scr): those that it would take by themselves, where
// their work together is worth its launches. The others keep the exact tiles. (Screening the whole batch where half of its scans by
// number allowed it, the rest redone after: a study of N = 1000, M = 3000 beside one of N = 4000, M = 20000 with an
// outlier took 13.5 ms; the exact tiles alone, and this rule, 12.0.)
bool batch_screen(const epi_batch *b, const epi_scan_params *p, std::vector<ScreenCut> &cut, std::vector<char> &scr)
{
    const size_t n = b->scans.size();
    cut.resize(n);
    scr.assign(n, 0);
    double work = 0.0;
    for (size_t s = 0; s < n; s++) {
        const Dataset &d = *b->data[b->scans[s].first];
        const int nchr = (int)d.chrstart.size();
        memset(&cut[s], 0, sizeof(ScreenCut));
        if (p->form != EPI_FORM_MFMA || !screen_fits(d) || !screen_cut(d.ph[b->scans[s].second], p, cut[s])) continue;
        scr[s] = 1;
        work += (double)block_pairs(d, 0, nchr * (nchr + 1) / 2) * d.nid * (d.missum[d.nsnp] ? 2.5 : 1.0);
    }
    if (work >= SCR_MIN_WORK) return true;
    scr.assign(n, 0);
    return false;
}

// Items of the next launch of a list through the screen, of `left`: as many as scr_chunk allows at the mean rate of each
// dataset's scans (the items of a dataset follow one another, tile by tile, each for every scan). (seg, used): the
// list's segment and the items taken from it.
int batch_chunk(const epi_batch *b, const std::vector<ScreenCut> &cut, int kind, int threads, int left, size_t &seg, long long &used)
{
    const int TA = b->scr_rows, TB = kind == 1 ? 32 : 64;
    int n = 0;
    double full = 0.0;  // part of a launch taken
    while (seg < b->segs[kind].size() && n < left) {
        const auto &s = b->segs[kind][seg];
        double rate = 0.0;
        int ns = 0;
        for (size_t i = 0; i < b->scans.size(); i++)
            if (b->scans[i].first == s.first && b->work_scr[i]) rate += cut[i].rate, ns++;
        const double most = scr_chunk(rate / ns, TA, TB, threads);
        const long long fit = (long long)((1.0 - full) * most), take = std::min(s.second - used, fit);
        n += (int)take;
        used += take;
        full += (double)take / most;
        if (used < s.second) break;
        seg++;
        used = 0;
    }
    // whole XCD groups: a few items more than a launch's share at most
    const int up = std::min(left, (n + 255) / 256 * 256);
    for (int more = up - n; more > 0 && seg < b->segs[kind].size();) {
        const int take = (int)std::min<long long>(more, b->segs[kind][seg].second - used);
        more -= take;
        if ((used += take) == b->segs[kind][seg].second) seg++, used = 0;
    }
    return up;
}

// Capture queue reset + the scan kernels as one graph: one kernel
// per list that has items (GENERAL and SPARSE first under order 1). Those of the exact tiles are persistent, with a grid
// of their occupancy times the CU count, so that every workgroup is resident and
// pulls work until its queues run dry; the screen's take a workgroup per item, each followed by resolve and redo.
int capture_batch(epi_batch *b, const epi_scan_params *p, const std::vector<ScreenCut> *cut)
{
    epi_ctx *c = b->ctx;
    drop_graph(b);
    if (cut) {
        HIPCHK(c, hipMemcpyAsync(b->d_cut, cut->data(), cut->size() * sizeof(ScreenCut), hipMemcpyHostToDevice, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    // The lists in the order of their launches: per kind the screened scans, then the others
    struct List {
        int kind, n, nt, grid;
        bool screen;
        const void *fn;
        BatchArgs B;
        ScreenBatchArgs G;
    };
    std::vector<List> lists;
    int Kl = 0;
    for (size_t s = 0; s < b->scans.size(); s++)
        if (b->work_scr[s]) Kl = std::max(Kl, (b->data[b->scans[s].first]->nid + KC - 1) / KC * KC);
    const int4 *work = b->d_work;
    uint32_t *redo = b->redo, *mask = b->mask;
    for (int l = 0; l < NLIST; l++) {
        const int kind = l % NKIND, n = (int)b->nlist[l];
        epi_schedule sg = b->work_sched;
        if (l < NKIND) sg.fast_rows = b->scr_rows;
        List L = {};
        L.kind = kind;
        L.n = n;
        L.screen = l < NKIND && !(kind == 2 && sg.dense_missing == 2);  // SPARSE tiles that the schedule asks for
        L.nt = L.screen ? 4 * sg.fast_rows : batch_threads_of(p->form, sg, kind);
        L.G = {b->d_mscan, b->d_cut, work, 0, 0, {c->cand, b->count->screen + 2 * kind, CAND_CAP, redo, mask}};
        L.B = {b->d_mscan, b->d_pscan, b->d_work, b->d_qpos + l * NQ, b->d_qend + l * NQ,
               make_sink(b->hits, &b->count->nhits, b->cap, p)};
        work += n;
        if (l < NKIND) {
            redo += batch_blocks(kind) * (size_t)n;
            mask += batch_blocks(kind) * (size_t)n;
        }
        if (!n) continue;
        L.fn = L.screen ? screen_batch_fn(sg, kind, batch_nocall(b)) : batch_kernel(p->form, sg, kind);
        int per_cu = 1;
        HIPCHK(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, L.fn, L.nt, 0));
        L.grid = std::max(1, per_cu) * c->ncu;
        lists.push_back(L);
    }
    // FAST, SPARSE, GENERAL; under order 1 GENERAL and SPARSE first
    static const int place[2][NKIND] = {{0, 2, 1}, {2, 0, 1}};
    const int *pl = place[b->work_sched.order == 1 ? 1 : 0];
    std::stable_sort(lists.begin(), lists.end(), [&](const List &x, const List &y) { return pl[x.kind] < pl[y.kind]; });
    epi_schedule scr_sched = b->work_sched;
    scr_sched.fast_rows = b->scr_rows;
    HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    hipLaunchKernelGGL(batch_reset, dim3(1), dim3(64), 0, c->stream, b->d_qpos, (const int *)b->d_qbegin, b->count);
    hipError_t le = hipGetLastError();
    for (List &L : lists) {
        if (le != hipSuccess) break;
        if (!L.screen) {
            void *args[] = {&L.B};
            le = hipLaunchKernel(L.fn, dim3(L.grid), dim3(L.nt), args, 0, c->stream);
            continue;
        }
        // one workgroup per item, a list of candidates at a time
        const int4 *items = L.G.work;
        const int halves = L.kind == 2 ? 2 : 1;
        ResolveArgs R = {{}, b->d_mscan, L.B.hs, c->cand, L.G.cs.count, CAND_CAP, resolve_lanes(Kl)};
        RedoArgs D = {{}, b->d_mscan, L.B.hs, items, L.G.cs.count, L.G.cs.redo, L.G.cs.mask};
        void *rargs[] = {&R}, *dargs[] = {&D};
        size_t seg = 0;
        long long used = 0;
        for (int t0 = 0; t0 < L.n && le == hipSuccess;) {
            if (t0) hipLaunchKernelGGL(empty_list, dim3(1), dim3(1), 0, c->stream, L.G.cs.count, CAND_CAP, &b->count->emptied);
            const int chunk = batch_chunk(b, *cut, L.kind, L.nt * halves, L.n - t0, seg, used);
            L.G.work = items + t0;
            L.G.item0 = t0;
            L.G.nitems = chunk;
            void *args[] = {&L.G};
            le = hipGetLastError();
            if (le == hipSuccess) le = hipLaunchKernel(L.fn, dim3(chunk * halves), dim3(L.nt), args, 0, c->stream);
            if (le == hipSuccess)
                le = hipLaunchKernel(L.kind ? (const void *)resolve_kernel<true, true> : (const void *)resolve_kernel<false, true>,
                                     dim3(4 * c->ncu), dim3(256), rargs, 0, c->stream);
            t0 += chunk;
        }
        if (le == hipSuccess)
            le = hipLaunchKernel(redo_batch_fn(scr_sched, L.kind), dim3(2 * c->ncu), dim3(256), dargs, 0, c->stream);
    }
    hipError_t ce = hipStreamEndCapture(c->stream, &b->graph);
    if (le != hipSuccess) return fail(c, EPI_ERR_HIP, "launch during capture: %s", hipGetErrorString(le));
    if (ce != hipSuccess) return fail(c, EPI_ERR_HIP, "hipStreamEndCapture: %s", hipGetErrorString(ce));
    HIPCHK(c, hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    b->gkey = *p;
    b->gvalid = true;
    b->gscreened = (int)std::count(b->work_scr.begin(), b->work_scr.end(), 1);
    b->grid = 0;
    for (const List &L : lists) b->grid = std::max(b->grid, L.grid);
    b->captures++;
    return EPI_OK;
}

// Work list and graph for (p, the batch's schedule of p->form), rebuilt only
// when the batch, the form, the schedule or the scan settings changed.
int batch_prepare(epi_batch *b, const epi_scan_params *p)
{
    int rc;
    if (p->form == EPI_FORM_MFMA)
        for (const auto &x : b->scans)
            if ((rc = check_mfma_phen(b->ctx, *b->data[x.first], x.second))) return rc;
    const epi_schedule &sc = b->sched[p->form];
    std::vector<ScreenCut> cut;
    std::vector<char> scr;
    const bool screen = batch_screen(b, p, cut, scr);
    int nid = 0;
    for (size_t s = 0; s < scr.size(); s++)
        if (scr[s]) nid = std::max(nid, b->data[b->scans[s].first]->nid);
    const int rows = screen_rows(nid);
    if (b->dirty || b->work_form != p->form || !same_schedule(b->work_sched, sc) || b->work_scr != scr || b->scr_rows != rows) {
        drop_graph(b);
        if ((rc = build_batch_work(b, p->form, sc, scr, rows))) return rc;
    }
    if (!b->gvalid || !same_key(b->gkey, *p))
        if ((rc = capture_batch(b, p, screen ? &cut : nullptr))) return rc;
    return EPI_OK;
}

// One replay of the captured graph; device time in ms.
int batch_run(epi_batch *b, double *ms_out)
{
    epi_ctx *c = b->ctx;
    b->dirty = true;  // a run that fails may leave marked blocks: the list is then built again
    HIPCHK(c, hipEventRecord(c->ev0, c->stream));
    HIPCHK(c, hipGraphLaunch(b->exec, c->stream));
    HIPCHK(c, hipEventRecord(c->ev1, c->stream));
    Counters n;
    HIPCHK(c, hipMemcpyAsync(&n, b->count, sizeof(n), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    float ms = 0.0f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    b->dirty = false;
    b->last_ms = ms;
    b->last_nhits = (long long)n.nhits;
    b->last_screened = b->gscreened;
    b->last_cand = candidates(n);
    b->last_redone = redone(n);
    b->fetched = false;
    if (ms_out) *ms_out = ms;
    return EPI_OK;
}

int batch_fetch(epi_batch *b)
{
    if (b->fetched) return EPI_OK;
    epi_ctx *c = b->ctx;
    long long have = std::min(b->last_nhits, b->cap);
    b->hh.resize((size_t)have);
    if (have) {
        HIPCHK(c, hipMemcpyAsync(b->hh.data(), b->hits, (size_t)have * sizeof(DevHit), hipMemcpyDeviceToHost,
                                 c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    b->by_scan.assign(b->scans.size(), {});
    for (long long t = 0; t < have; t++) {
        int s = b->hh[t].tag;
        if (s >= 0 && s < (int)b->scans.size()) b->by_scan[s].push_back((int)t);
    }
    b->fetched = true;
    return EPI_OK;
}

// Clears the counters (hits: that of the hits too) and, before the screen first runs over a tile list, the masks of its blocks.
int reset_scan(epi_ctx *c, bool hits, bool screen)
{
    constexpr uint32_t words = sizeof(Counters) / sizeof(uint32_t), first = offsetof(Counters, screen) / sizeof(uint32_t);
    const size_t n = screen && !c->masks_set ? c->redo_blocks : 0;
    hipLaunchKernelGGL(clear_words, dim3((unsigned)(n / 256 + 1)), dim3(n ? 256 : 64), 0, c->stream,
                       reinterpret_cast<uint32_t *>(c->count), hits ? 0u : first, words, c->redo + c->redo_blocks, n);
    HIPCHK(c, hipGetLastError());
    if (screen) c->masks_set = true;
    return EPI_OK;
}

// One scan of the block range of p with schedule sc: tile list, upload,
// pair kernels, hit count. Records the device time and counts in c. A tile
// list of up to c->max_tiles tiles is built once and kept on the device; a
// longer one is built, uploaded and launched in pieces of about that many
// tiles, and the timed region then also holds the uploads of the later pieces.
int run_scan(epi_ctx *c, const epi_scan_params *p, const epi_schedule &asked)
{
    int rc;
    int nchr = (int)c->d.chrstart.size();
    int nblk = nchr * (nchr + 1) / 2;
    int bb = std::max(0, p->blk_begin), be = p->blk_end <= 0 ? nblk : std::min(nblk, p->blk_end);
    ScreenCut cut;
    const bool screen = screened(c->d, p, block_pairs(c->d, bb, be), cut);
    epi_schedule sc = asked;
    if (screen) sc.fast_rows = screen_rows(c->d.nid);
    const size_t max_tiles = screen ? scr_piece(c->max_tiles) : c->max_tiles;
    TileLists &tl = c->tl;
    const bool cached = c->tl_valid && c->tl_bb == bb && c->tl_be == be && c->tl_form == p->form &&
                        same_schedule(c->tl_sched, sc) && (!screen || c->redo);
    TileCursor cur;
    cur.blk = bb;
    bool done = cached;
    if (!cached) {
        tl = TileLists();
        done = build_tiles(c->d, be, p->form, sc, max_tiles, cur, tl);
        if ((rc = upload_tiles(c, tl, screen))) return rc;
        c->tl_bb = bb;
        c->tl_be = be;
        c->tl_form = p->form;
        c->tl_sched = sc;
    }
    const bool whole = done;  // the list serves later scans
    c->tl_valid = false;  // a scan that fails may leave marked blocks
    if ((rc = reset_scan(c, true, screen))) return rc;
    DumpSink ds;
    memset(&ds, 0, sizeof(ds));
    HIPCHK(c, hipEventRecord(c->ev0, c->stream));
    long long pairs = tl.pairs;
    c->last_tiles[0] = c->last_tiles[1] = c->last_tiles[2] = 0;
    c->last_digits = screen ? cut.nd : 0;
    c->last_cand = c->last_redone = 0;
    int launches = 0;
    Counters n;
    for (;;) {
        if ((rc = launch_pairs<false>(c, p, sc, tl, ds, ctx_bufs(c), screen ? &cut : nullptr))) return rc;
        launches += c->last_launches;
        HIPCHK(c, hipEventRecord(c->ev1, c->stream));
        // the launched kernels read the device tile list that the next piece overwrites
        HIPCHK(c, hipMemcpyAsync(&n, c->count, sizeof(n), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        c->last_cand += candidates(n);
        c->last_redone += redone(n);
        if (redone(n)) {
            // few scans have blocks to redo: launched for every kind in every scan, N = 500, M = 2000 took 102.7 us, not 100.6
            if ((rc = launch_pairs<false>(c, p, sc, tl, ds, ctx_bufs(c), &cut, n.screen))) return rc;
            launches += c->last_launches;
            HIPCHK(c, hipEventRecord(c->ev1, c->stream));
            HIPCHK(c, hipMemcpyAsync(&n, c->count, sizeof(n), hipMemcpyDeviceToHost, c->stream));
            HIPCHK(c, hipStreamSynchronize(c->stream));
        }
        if (done) break;
        tl = TileLists();
        done = build_tiles(c->d, be, p->form, sc, max_tiles, cur, tl);
        if ((rc = upload_tiles(c, tl, screen))) return rc;
        if ((rc = reset_scan(c, false, screen))) return rc;
        pairs += tl.pairs;
    }
    float ms = 0.0f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->tl_valid = whole;
    c->last_ms = ms;
    c->last_pairs = pairs;
    c->last_launches = launches;
    c->last_nhits = (long long)n.nhits;
    return EPI_OK;
}

// Coordinate descent over the schedule dimensions in `dims`: each dimension
// in turn is set to every candidate value (others fixed at the best so far)
// and the fastest is kept. measure(s, ms) times one schedule; repeated
// schedules are timed once. Candidates that measure equal keep the earlier.
template <class Measure>
int tune_descent(int form, int dims, epi_schedule &cur, double &tcur, int &nmeasured, epi_tune_entry *log,
                 int log_cap, Measure measure)
{
    std::vector<std::pair<epi_schedule, double>> seen;
    auto timed = [&](const epi_schedule &s, double &ms) -> int {
        for (auto &e : seen)
            if (same_schedule(e.first, s)) {
                ms = e.second;
                return EPI_OK;
            }
        int r = measure(s, ms);
        if (r) return r;
        seen.push_back({s, ms});
        if (log && nmeasured < log_cap) {
            log[nmeasured].sched = s;
            log[nmeasured].ms = ms;
        }
        nmeasured++;
        return EPI_OK;
    };
    int rc = timed(cur, tcur);
    if (rc) return rc;
    auto tryit = [&](const epi_schedule &s) -> int {
        double t = 0.0;
        int r = timed(s, t);
        if (r) return r;
        if (t < tcur) {
            cur = s;
            tcur = t;
        }
        return EPI_OK;
    };
    const int rows_m[] = {32, 64}, rows_p[] = {32, 16};
    const int sup[][2] = {{8, 4}, {4, 4}, {16, 2}, {4, 8}, {1, 1}};
    if ((dims & EPI_TUNE_MISSING) && form == EPI_FORM_MFMA)
        for (int v : {0, 1, 2}) {
            epi_schedule s = cur;
            s.dense_missing = v;
            if ((rc = tryit(s))) return rc;
        }
    if (dims & EPI_TUNE_ROWS)
        for (int v : (form == EPI_FORM_MFMA ? rows_m : rows_p)) {
            epi_schedule s = cur;
            s.fast_rows = v;
            if ((rc = tryit(s))) return rc;
        }
    if (dims & EPI_TUNE_SUPER)
        for (auto &v : sup) {
            epi_schedule s = cur;
            s.super_a = v[0];
            s.super_b = v[1];
            if ((rc = tryit(s))) return rc;
        }
    if (dims & EPI_TUNE_QUEUES)
        for (int v : {8, 1}) {
            epi_schedule s = cur;
            s.queues = v;
            if ((rc = tryit(s))) return rc;
        }
    if (dims & EPI_TUNE_ORDER)
        for (int v : {0, 1, 2}) {
            epi_schedule s = cur;
            s.order = v;
            if ((rc = tryit(s))) return rc;
        }
    return EPI_OK;
}

}  // namespace

// ============================================================== C ABI ====

extern "C" {

const char *epi_strerror(int code)
{
    switch (code) {
    case EPI_OK: return "ok";
    case EPI_ERR_ARG: return "invalid argument";
    case EPI_ERR_HIP: return "HIP runtime error";
    case EPI_ERR_NODEV: return "no such device";
    case EPI_ERR_STATE: return "required data not set";
    case EPI_ERR_NOMEM: return "device out of memory";
    case EPI_ERR_RANGE: return "value out of range";
    default: return "unknown error";
    }
}

const char *epi_last_error(const epi_ctx *c) { return c ? c->err.c_str() : "null context"; }

int epi_open(int device, epi_ctx **out)
{
    if (!out) return EPI_ERR_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return EPI_ERR_NODEV;
    if (device < 0 || device >= n) return EPI_ERR_NODEV;
    epi_ctx *c = new epi_ctx();
    c->device = device;
    if (hipSetDevice(device) != hipSuccess ||
        hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
        delete c;
        return EPI_ERR_HIP;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) {
        snprintf(c->name, sizeof(c->name), "%s (%s, %d CUs)", prop.name, prop.gcnArchName, prop.multiProcessorCount);
        c->ncu = prop.multiProcessorCount;
    }
    if (c->ncu <= 0) c->ncu = 1;
    for (int f = 0; f < 2; f++) c->sched[f] = default_schedule(f);
    if (dalloc(c, c->count, 1) || dalloc(c, c->hits, (size_t)c->cap) || dalloc(c, c->cand, (size_t)CAND_CAP)) {
        epi_close(c);
        return EPI_ERR_NOMEM;
    }
    if (scratch_of(c, &c->scratch)) {
        epi_close(c);
        return EPI_ERR_HIP;
    }
    *out = c;
    return EPI_OK;
}

void epi_close(epi_ctx *c)
{
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_dataset(c->d);
    dfree(c->hits);
    dfree(c->count);
    dfree(c->tiles);
    dfree(c->cand);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

int epi_device_name(const epi_ctx *c, char *buf, size_t n)
{
    if (!c || !buf || n == 0) return EPI_ERR_ARG;
    snprintf(buf, n, "%s", c->name);
    return EPI_OK;
}

// Marginals as soon as genotypes and phenotypes are both set, so that scans
// (epi_scan_noalloc among them) find them ready. A failure drops the
// phenotypes.
int ready_marginals(epi_ctx *c)
{
    if (!c->d.mbits || c->d.ph.empty()) return EPI_OK;
    const int rc = ds_marginals(c, c->d);
    if (rc) drop_phenotypes(c->d);
    return rc;
}

int epi_set_genotypes(epi_ctx *c, const int32_t *words, int32_t nid, int32_t nsnp)
{
    if (!c) return EPI_ERR_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    c->last_nhits = 0;
    c->tl_valid = false;
    int rc = ds_set_genotypes(c, c->d, words, nid, nsnp);
    if (!rc) rc = ds_sparse(c, c->d);
    return rc ? rc : ready_marginals(c);
}

int epi_set_phenotypes_ex(epi_ctx *c, const float *phen, int32_t nphen, int32_t nid, int32_t flags)
{
    if (!c) return EPI_ERR_ARG;
    if (flags & ~EPI_PHEN_NINE_IS_VALUE) return fail(c, EPI_ERR_ARG, "unknown phenotype flags");
    HIPCHK(c, hipSetDevice(c->device));
    const int rc = ds_set_phenotypes(c, c->d, phen, nphen, nid, flags);
    return rc ? rc : ready_marginals(c);
}

int epi_set_phenotypes(epi_ctx *c, const float *phen, int32_t nphen, int32_t nid)
{
    return epi_set_phenotypes_ex(c, phen, nphen, nid, 0);
}

int epi_phen_encoding(const float *phen, int32_t nid, int32_t flags, epi_phen_info *info)
{
    if (!phen || !info || nid < 2 || nid > MAX_NID || (flags & ~EPI_PHEN_NINE_IS_VALUE)) return EPI_ERR_ARG;
    PhenEnc e;
    const int Kp = (nid + KPAD - 1) / KPAD * KPAD;
    const int rc = encode_phen(nullptr, phen, nid, Kp, (flags & EPI_PHEN_NINE_IS_VALUE) != 0, 0, false, e);
    if (rc) return rc;
    memset(info, 0, sizeof(*info));
    info->present = e.p.nV;
    info->outliers = e.p.nout;
    info->mfma_ok = e.p.mfma_ok ? 1 : 0;
    info->fbits = e.p.fbits;
    info->zbits = e.p.zbits;
    info->centre = e.p.centre;
    info->central_sd = e.p.sc;
    info->max_dev = e.p.maxdev;
    for (int t = 0; t < e.p.nout; t++) info->outlier_index[t] = e.oidx[t];
    return EPI_OK;
}

int epi_set_chromosomes(epi_ctx *c, const int32_t *chrstart, const int32_t *chrsize, int32_t nchr)
{
    if (!c) return EPI_ERR_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    c->tl_valid = false;
    int rc = ds_set_chromosomes(c, c->d, chrstart, chrsize, nchr);
    if (!rc) rc = ds_sparse(c, c->d);
    return rc;
}

void epi_scan_params_default(epi_scan_params *p)
{
    if (!p) return;
    memset(p, 0, sizeof(*p));
    p->test = 'f';
    p->form = EPI_FORM_MFMA;
    p->t1 = 6.5f;
    p->t2 = 10.5f;
    p->phen = 0;
    p->blk_begin = 0;
    p->blk_end = 0;
}

int epi_set_hit_capacity(epi_ctx *c, int64_t cap)
{
    if (!c || cap < 1) return EPI_ERR_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    c->cap = c->last_nhits = 0;  // a failure leaves no buffer: scans then count their hits and report the overflow
    int rc = dalloc(c, c->hits, (size_t)cap);
    if (rc) return rc;
    c->cap = cap;
    return EPI_OK;
}

int epi_set_max_tiles(epi_ctx *c, int64_t max_tiles)
{
    if (!c || max_tiles < 1 || max_tiles > (int64_t)INT32_MAX / 2) return EPI_ERR_ARG;
    c->max_tiles = (size_t)max_tiles;
    c->tl_valid = false;
    return EPI_OK;
}

int epi_scan(epi_ctx *c, const epi_scan_params *p)
{
    if (!c) return EPI_ERR_ARG;
    int rc = check_params(c, p);
    if (rc) return rc;
    HIPCHK(c, hipSetDevice(c->device));
    if ((rc = ds_marginals(c, c->d))) return rc;
    return run_scan(c, p, c->sched[p->form]);
}

int epi_scan_noalloc(epi_ctx *c, const epi_scan_params *p, epi_hit64 *hits, int64_t cap, int64_t *nhits)
{
    if (!c) return EPI_ERR_ARG;
    int rc = check_params(c, p);
    if (rc) return rc;
    if (!hits || cap < 0 || !nhits) return fail(c, EPI_ERR_ARG, "need a device hit buffer, its capacity and nhits");
    if (!c->d.marg_ok) return fail(c, EPI_ERR_STATE, "genotypes and phenotypes must both be set");
    if (!c->scratch) return fail(c, EPI_ERR_STATE, "no scratch address for this device");
    HIPCHK(c, hipSetDevice(c->device));
    const epi_schedule &sc = c->sched[p->form];
    const int nchr = (int)c->d.chrstart.size(), nblk = nchr * (nchr + 1) / 2;
    const int bb = std::max(0, p->blk_begin), be = p->blk_end <= 0 ? nblk : std::min(nblk, p->blk_end);
    TileLists tl;
    TileCursor cur;
    cur.blk = bb;
    const bool done = build_tiles(c->d, be, p->form, sc, NOALLOC_TILES + 1, cur, tl);
    const size_t nt = tl.count();
    if (!done || nt > NOALLOC_TILES)
        return fail(c, EPI_ERR_RANGE,
                    "the scan needs more than the %zu tiles the no-allocation scratch holds (%zu MiB); use epi_scan",
                    NOALLOC_TILES, NOALLOC_BYTES >> 20);
    unsigned char *base = static_cast<unsigned char *>(c->scratch);
    const ScanBufs B = {reinterpret_cast<int4 *>(base + 256), reinterpret_cast<DevHit *>(hits),
                        reinterpret_cast<unsigned long long *>(base), (long long)cap, {}};
    if ((rc = copy_tiles(c, B.tiles, tl))) return rc;
    c->last_tiles[0] = c->last_tiles[1] = c->last_tiles[2] = 0;
    hipLaunchKernelGGL(zero_counter, dim3(1), dim3(1), 0, c->stream, B.nhits);
    HIPCHK(c, hipGetLastError());
    DumpSink ds;
    memset(&ds, 0, sizeof(ds));
    HIPCHK(c, hipEventRecord(c->ev0, c->stream));
    if ((rc = launch_pairs<false>(c, p, sc, tl, ds, B))) return rc;
    HIPCHK(c, hipEventRecord(c->ev1, c->stream));
    unsigned long long nh = 0;
    HIPCHK(c, hipMemcpyAsync(&nh, B.nhits, sizeof(nh), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    float ms = 0.0f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    c->last_pairs = tl.pairs;
    *nhits = (int64_t)nh;
    return EPI_OK;
}

int epi_autotune(epi_ctx *c, const epi_scan_params *p, int32_t dims, int32_t reps, epi_schedule *best,
                 double *best_ms, epi_tune_entry *log, int32_t log_cap, int32_t *nlog)
{
    if (!c) return EPI_ERR_ARG;
    int rc = check_params(c, p);
    if (rc) return rc;
    if (reps < 1 || reps > 100) return fail(c, EPI_ERR_ARG, "reps must be in [1, 100]");
    // queues and order do not apply to single scans; the missing-call tiles only with missing calls
    const bool anymiss = !c->d.missc.empty() && c->d.missc[c->d.nsnp] > 0;
    if (dims == 0) dims = EPI_TUNE_ROWS | EPI_TUNE_SUPER | (anymiss ? EPI_TUNE_MISSING : 0);
    dims &= EPI_TUNE_ROWS | EPI_TUNE_SUPER | EPI_TUNE_MISSING;
    HIPCHK(c, hipSetDevice(c->device));
    if ((rc = ds_marginals(c, c->d))) return rc;
    // a screened scan picks its tile height itself: the value for other scans is not to be had from its times
    const int nchr = (int)c->d.chrstart.size(), nblk = nchr * (nchr + 1) / 2;
    ScreenCut cut;
    if (screened(c->d, p, block_pairs(c->d, std::max(0, p->blk_begin), p->blk_end <= 0 ? nblk : std::min(nblk, p->blk_end)), cut))
        dims &= ~EPI_TUNE_ROWS;
    epi_schedule cur = c->sched[p->form];
    double tcur = 0.0;
    int n = 0;
    rc = tune_descent(p->form, dims, cur, tcur, n, log, log_cap, [&](const epi_schedule &s, double &ms) -> int {
        int r = run_scan(c, p, s);  // warm-up
        if (r) return r;
        std::vector<double> t(reps);
        for (int i = 0; i < reps; i++) {
            if ((r = run_scan(c, p, s))) return r;
            t[i] = c->last_ms;
        }
        std::sort(t.begin(), t.end());
        ms = t[reps / 2];
        return EPI_OK;
    });
    if (rc) return rc;
    c->sched[p->form] = cur;
    if (best) *best = cur;
    if (best_ms) *best_ms = tcur;
    if (nlog) *nlog = n;
    return EPI_OK;
}

int epi_hit_count(epi_ctx *c, int64_t *nhits, int32_t *overflow)
{
    if (!c) return EPI_ERR_ARG;
    if (nhits) *nhits = c->last_nhits;
    if (overflow) *overflow = c->last_nhits > c->cap;
    return EPI_OK;
}

int epi_get_hits(epi_ctx *c, epi_hit *hits, double *F64, double *F2_64, int32_t *block, int64_t cap, int64_t *n)
{
    if (!c || cap < 0) return EPI_ERR_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    long long have = std::min<long long>(c->last_nhits, c->cap);
    const std::unique_ptr<DevHit[]> h(new DevHit[(size_t)have]);  // not cleared
    if (have) {
        HIPCHK(c, hipMemcpyAsync(h.get(), c->hits, (size_t)have * sizeof(DevHit), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    std::vector<int> idx((size_t)have);
    for (long long t = 0; t < have; t++) idx[t] = (int)t;
    long long m = 0;
    emit_hits(c->d, h.get(), idx, hits, F64, F2_64, block, cap, &m);
    if (n) *n = m;
    return EPI_OK;
}

int epi_set_schedule(epi_ctx *c, int32_t form, const epi_schedule *s)
{
    if (!c || !s || (form != EPI_FORM_PLAIN && form != EPI_FORM_MFMA)) return EPI_ERR_ARG;
    if (!valid_schedule(form, *s)) return fail(c, EPI_ERR_ARG, "invalid schedule for this form");
    c->sched[form] = *s;
    return EPI_OK;
}

int epi_get_schedule(epi_ctx *c, int32_t form, epi_schedule *s)
{
    if (!c || !s || (form != EPI_FORM_PLAIN && form != EPI_FORM_MFMA)) return EPI_ERR_ARG;
    *s = c->sched[form];
    return EPI_OK;
}

int epi_last_scan_stats(epi_ctx *c, double *kernel_ms, int64_t *pairs, int32_t *launches)
{
    if (!c) return EPI_ERR_ARG;
    if (kernel_ms) *kernel_ms = c->last_ms;
    if (pairs) *pairs = c->last_pairs;
    if (launches) *launches = c->last_launches;
    return EPI_OK;
}

int epi_last_tiles(epi_ctx *c, int64_t *fast, int64_t *sparse, int64_t *general)
{
    if (!c) return EPI_ERR_ARG;
    if (fast) *fast = c->last_tiles[0];
    if (sparse) *sparse = c->last_tiles[1];
    if (general) *general = c->last_tiles[2];
    return EPI_OK;
}

int epi_last_screen(epi_ctx *c, int32_t *digits, int64_t *candidates, int64_t *redone)
{
    if (!c) return EPI_ERR_ARG;
    if (digits) *digits = c->last_digits;
    if (candidates) *candidates = c->last_cand;
    if (redone) *redone = c->last_redone;
    return EPI_OK;
}

int epi_pair_dump(epi_ctx *c, const epi_scan_params *p, int32_t a0, int32_t a1, int32_t b0, int32_t b1,
                  int32_t *counts, double *sums, double *F, double *F2)
{
    if (!c) return EPI_ERR_ARG;
    int rc = check_params(c, p);
    if (rc) return rc;
    if (a0 < 0 || b0 < 0 || a1 > c->d.nsnp || b1 > c->d.nsnp || a1 <= a0 || b1 <= b0)
        return fail(c, EPI_ERR_ARG, "dump rectangle out of range");
    HIPCHK(c, hipSetDevice(c->device));
    if ((rc = ds_marginals(c, c->d))) return rc;
    const epi_schedule &sc = c->sched[p->form];
    const int TA = sc.fast_rows, TB = TILE_B;
    // Tiles over the rectangle in global SNP space (no block restriction). A
    // tile can be SPARSE where its a- and b-ranges each lie in one chromosome
    // and start on the virtual word grid, as every tile of a scan does.
    const Dataset &d = c->d;
    const bool sp = use_sparse(d, p->form, sc);
    std::vector<int32_t> vidx;
    if (sp) virtual_order(d, vidx, nullptr);
    auto grid = [&](int s0, int s1, int w) {
        const int ch = d.snpchr[s0];
        return ch >= 0 && d.snpchr[s1 - 1] == ch && vidx[s0] % w == 0;
    };
    TileLists all;
    for (int x = a0; x < a1; x += TA)
        for (int y = b0; y < b1; y += TB) {
            const int x1 = std::min(a1, x + TA), y1 = std::min(b1, y + TB);
            emit_tile(d, x, x1, y, y1, gen_rows(p->form, sc), gen_cols(p->form, sc),
                      sp && grid(x, x1, TA) && grid(y, y1, 64), sc.dense_missing == 2, all);
        }
    if ((rc = upload_tiles(c, all, false))) return rc;
    long long np = (long long)(a1 - a0) * (b1 - b0);
    int32_t *dc = nullptr;
    double *dsum = nullptr, *dF = nullptr, *dF2 = nullptr;
    if ((rc = dalloc(c, dc, (size_t)np * 9)) || (rc = dalloc(c, dsum, (size_t)np * 9)) ||
        (rc = dalloc(c, dF, (size_t)np)) || (rc = dalloc(c, dF2, (size_t)np))) {
        dfree(dc);
        dfree(dsum);
        dfree(dF);
        return rc;
    }
    DumpSink ds;
    ds.counts = dc;
    ds.sums = dsum;
    ds.F = dF;
    ds.F2 = dF2;
    ds.a0 = a0;
    ds.a1 = a1;
    ds.b0 = b0;
    ds.b1 = b1;
    const PhenDev &ph = c->d.ph[p->phen];
    ds.unit = p->form == EPI_FORM_MFMA ? std::ldexp(1.0, -ph.fbits) : std::ldexp(1.0, ph.ybits);
    ds.centre = ph.centre;
    // Pre-fill with the caller's buffers so that pairs with a <= b keep their values.
    int hrc = EPI_OK;
    auto h2d = [&](void *d, const void *hsrc, size_t bytes) {
        if (hrc == EPI_OK && hsrc && hipMemcpyAsync(d, hsrc, bytes, hipMemcpyHostToDevice, c->stream) != hipSuccess)
            hrc = fail(c, EPI_ERR_HIP, "dump prefill copy failed");
    };
    h2d(dc, counts, (size_t)np * 9 * 4);
    h2d(dsum, sums, (size_t)np * 9 * 8);
    h2d(dF, F, (size_t)np * 8);
    h2d(dF2, F2, (size_t)np * 8);
    c->last_tiles[0] = c->last_tiles[1] = c->last_tiles[2] = 0;
    if (hrc == EPI_OK) hrc = launch_pairs<true>(c, p, sc, all, ds, ctx_bufs(c));
    auto d2h = [&](void *hdst, const void *d, size_t bytes) {
        if (hrc == EPI_OK && hdst && hipMemcpyAsync(hdst, d, bytes, hipMemcpyDeviceToHost, c->stream) != hipSuccess)
            hrc = fail(c, EPI_ERR_HIP, "dump copy back failed");
    };
    d2h(counts, dc, (size_t)np * 9 * 4);
    d2h(sums, dsum, (size_t)np * 9 * 8);
    d2h(F, dF, (size_t)np * 8);
    d2h(F2, dF2, (size_t)np * 8);
    if (hrc == EPI_OK && hipStreamSynchronize(c->stream) != hipSuccess) hrc = fail(c, EPI_ERR_HIP, "dump sync failed");
    dfree(dc);
    dfree(dsum);
    dfree(dF);
    dfree(dF2);
    return hrc;
}

int epi_screen_dump(epi_ctx *c, const epi_scan_params *p, int32_t digits, int32_t a0, int32_t a1, int32_t b0, int32_t b1,
                    int32_t *v, float *counts, float *sums)
{
    if (!c) return EPI_ERR_ARG;
    int rc = check_params(c, p);
    if (rc) return rc;
    if (p->form != EPI_FORM_MFMA || digits < 1 || digits > 2 || !counts || !sums)
        return fail(c, EPI_ERR_ARG, "the MFMA form, one or two digits, and both outputs");
    const Dataset &d = c->d;
    if (a0 < 0 || b0 < 0 || a1 > d.nsnp || b1 > d.nsnp || a1 <= a0 || b1 <= b0)
        return fail(c, EPI_ERR_ARG, "dump rectangle out of range");
    const PhenDev &ph = d.ph[p->phen];
    if (!planes_fit(d) || !(ph.scr[digits - 1].delta > 0.0))
        return fail(c, EPI_ERR_RANGE, "the screen does not take this dataset or phenotype");
    HIPCHK(c, hipSetDevice(c->device));
    if ((rc = ds_marginals(c, c->d))) return rc;
    const int TA = screen_rows(d.nid);
    TileLists all;
    for (int x = a0; x < a1; x += TA)
        for (int y = b0; y < b1; y += TILE_B) emit_tile(d, x, std::min(a1, x + TA), y, std::min(b1, y + TILE_B), TA, 32, false, false, all);
    if (all.count() >= 1u << 23) return fail(c, EPI_ERR_ARG, "dump rectangle too large");  // one launch of 256-thread tiles
    if ((rc = upload_tiles(c, all, false))) return rc;
    const size_t n = (size_t)(a1 - a0) * (b1 - b0) * 9;
    float *out = nullptr;
    if ((rc = dalloc(c, out, 2 * n))) return rc;
    ScreenArgs A;
    memset(&A, 0, sizeof(A));
    A.S = mfma_scan(d, p->phen, p->phen);
    A.cut.N = (float)(ph.nV / 64.0);
    A.cut.vs = (float)(ph.scr[digits - 1].vsum / 64.0);
    const ScreenDump D = {out, out + n, a0, b0, b1 - b0};
    const bool nocall = TA == 64 && scr_nocall(A.S.Kl);
    hipError_t he = hipMemsetAsync(out, 0xFF, 2 * n * sizeof(float), c->stream);  // NaN
    auto launch = [&](auto kernel, const int4 *tiles, size_t nt) {
        if (he != hipSuccess || !nt) return;
        A.tiles = tiles;
        A.ntiles = (int)nt;
        hipLaunchKernelGGL(kernel, dim3((unsigned)nt), dim3(4 * TA), 0, c->stream, A, D);
        he = hipGetLastError();
    };
    const size_t nf = all.fast.size(), ng = all.gen.size();
    if (TA == 64) {
        launch(digits == 1 ? screen_fast_dump<64, 1> : screen_fast_dump<64, 2>, c->tiles, nf);
        if (nocall) launch(digits == 1 ? screen_gen_dump<64, 1, true> : screen_gen_dump<64, 2, true>, c->tiles + nf, ng);
        else launch(digits == 1 ? screen_gen_dump<64, 1, false> : screen_gen_dump<64, 2, false>, c->tiles + nf, ng);
    } else {
        launch(digits == 1 ? screen_fast_dump<32, 1> : screen_fast_dump<32, 2>, c->tiles, nf);
        launch(digits == 1 ? screen_gen_dump<32, 1, false> : screen_gen_dump<32, 2, false>, c->tiles + nf, ng);
    }
    std::vector<MissPhen> mp(v ? d.nid : 0);
    if (he == hipSuccess) he = hipMemcpyAsync(counts, out, n * sizeof(float), hipMemcpyDeviceToHost, c->stream);
    if (he == hipSuccess) he = hipMemcpyAsync(sums, out + n, n * sizeof(float), hipMemcpyDeviceToHost, c->stream);
    if (he == hipSuccess && v) he = hipMemcpyAsync(mp.data(), ph.mp, mp.size() * sizeof(MissPhen), hipMemcpyDeviceToHost, c->stream);
    if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
    dfree(out);
    if (he != hipSuccess) return fail(c, EPI_ERR_HIP, "screen dump: %s", hipGetErrorString(he));
    for (size_t k = 0; k < mp.size(); k++) v[k] = mp[k].sv[digits - 1];
    return EPI_OK;
}

// ------------------------------------------------------------------ batch --

int epi_batch_create(epi_ctx *c, epi_batch **out)
{
    if (!c || !out) return EPI_ERR_ARG;
    *out = nullptr;
    HIPCHK(c, hipSetDevice(c->device));
    epi_batch *b = new epi_batch();
    b->ctx = c;
    c->batches.push_back(b);
    for (int f = 0; f < 2; f++) b->sched[f] = default_schedule(f);
    int rc;
    if ((rc = dalloc(c, b->d_qpos, NLIST * NQ)) || (rc = dalloc(c, b->d_qbegin, NLIST * NQ)) ||
        (rc = dalloc(c, b->d_qend, NLIST * NQ)) ||
        (rc = dalloc(c, b->count, 1)) || (rc = dalloc(c, b->hits, (size_t)b->cap))) {
        epi_batch_destroy(b);
        return rc;
    }
    *out = b;
    return EPI_OK;
}

void epi_batch_destroy(epi_batch *b)
{
    if (!b) return;
    epi_ctx *c = b->ctx;
    c->batches.erase(std::remove(c->batches.begin(), c->batches.end(), b), c->batches.end());
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    drop_graph(b);
    for (Dataset *d : b->data) {
        free_dataset(*d);
        delete d;
    }
    dfree(b->d_mscan);
    dfree(b->d_pscan);
    dfree(b->d_cut);
    dfree(b->d_work);
    dfree(b->d_qpos);
    dfree(b->d_qbegin);
    dfree(b->d_qend);
    dfree(b->hits);
    dfree(b->count);
    delete b;
}

int epi_batch_add_dataset(epi_batch *b, const int32_t *words, int32_t nid, int32_t nsnp, const int32_t *chrstart,
                          const int32_t *chrsize, int32_t nchr, int32_t *dataset)
{
    if (!b) return EPI_ERR_ARG;
    epi_ctx *c = b->ctx;
    HIPCHK(c, hipSetDevice(c->device));
    Dataset *d = new Dataset();
    int rc = ds_set_genotypes(c, *d, words, nid, nsnp);
    if (!rc && chrstart) rc = ds_set_chromosomes(c, *d, chrstart, chrsize, nchr);
    if (!rc) rc = ds_sparse(c, *d);
    if (rc) {
        free_dataset(*d);
        delete d;
        return rc;
    }
    b->data.push_back(d);
    b->dirty = true;
    if (dataset) *dataset = (int32_t)b->data.size() - 1;
    return EPI_OK;
}

int epi_batch_add_phenotypes(epi_batch *b, int32_t dataset, const float *phen, int32_t nphen, int32_t *first_scan)
{
    return epi_batch_add_phenotypes_ex(b, dataset, phen, nphen, 0, first_scan);
}

int epi_batch_add_phenotypes_ex(epi_batch *b, int32_t dataset, const float *phen, int32_t nphen, int32_t flags,
                                int32_t *first_scan)
{
    if (!b) return EPI_ERR_ARG;
    epi_ctx *c = b->ctx;
    if (flags & ~EPI_PHEN_NINE_IS_VALUE) return fail(c, EPI_ERR_ARG, "unknown phenotype flags");
    if (dataset < 0 || dataset >= (int)b->data.size()) return fail(c, EPI_ERR_ARG, "no such dataset");
    Dataset &d = *b->data[dataset];
    if (!d.ph.empty()) return fail(c, EPI_ERR_STATE, "dataset %d already has phenotypes", dataset);
    HIPCHK(c, hipSetDevice(c->device));
    int rc = ds_set_phenotypes(c, d, phen, nphen, d.nid, flags);
    if (!rc) rc = ds_marginals(c, d);
    if (rc) {
        drop_phenotypes(d);
        return rc;
    }
    if (first_scan) *first_scan = (int32_t)b->scans.size();
    for (int r = 0; r < nphen; r++) b->scans.push_back({dataset, r});
    b->dirty = true;
    return EPI_OK;
}

int epi_batch_set_hit_capacity(epi_batch *b, int64_t cap)
{
    if (!b || cap < 1) return EPI_ERR_ARG;
    epi_ctx *c = b->ctx;
    HIPCHK(c, hipSetDevice(c->device));
    drop_graph(b);  // it holds the old buffer
    b->cap = b->last_nhits = 0;  // as epi_set_hit_capacity
    b->fetched = false;
    int rc = dalloc(c, b->hits, (size_t)cap);
    if (rc) return rc;
    b->cap = cap;
    return EPI_OK;
}

int epi_batch_scan(epi_batch *b, const epi_scan_params *p)
{
    if (!b) return EPI_ERR_ARG;
    epi_ctx *c = b->ctx;
    int rc = check_common(c, p);
    if (rc) return rc;
    if (b->scans.empty()) return fail(c, EPI_ERR_STATE, "batch has no scans");
    HIPCHK(c, hipSetDevice(c->device));
    if ((rc = batch_prepare(b, p))) return rc;
    return batch_run(b, nullptr);
}

int epi_batch_set_schedule(epi_batch *b, int32_t form, const epi_schedule *s)
{
    if (!b || !s || (form != EPI_FORM_PLAIN && form != EPI_FORM_MFMA)) return EPI_ERR_ARG;
    if (!valid_schedule(form, *s)) return fail(b->ctx, EPI_ERR_ARG, "invalid schedule for this form");
    b->sched[form] = *s;
    return EPI_OK;
}

int epi_batch_get_schedule(epi_batch *b, int32_t form, epi_schedule *s)
{
    if (!b || !s || (form != EPI_FORM_PLAIN && form != EPI_FORM_MFMA)) return EPI_ERR_ARG;
    *s = b->sched[form];
    return EPI_OK;
}

int epi_batch_autotune(epi_batch *b, const epi_scan_params *p, int32_t dims, int32_t reps, epi_schedule *best,
                       double *best_ms, epi_tune_entry *log, int32_t log_cap, int32_t *nlog)
{
    if (!b) return EPI_ERR_ARG;
    epi_ctx *c = b->ctx;
    int rc = check_common(c, p);
    if (rc) return rc;
    if (b->scans.empty()) return fail(c, EPI_ERR_STATE, "batch has no scans");
    if (reps < 1 || reps > 100) return fail(c, EPI_ERR_ARG, "reps must be in [1, 100]");
    if (dims == 0) dims = EPI_TUNE_ALL;
    HIPCHK(c, hipSetDevice(c->device));
    const int form = p->form;
    // the tile height and the queues are those of scans that are not screened
    std::vector<ScreenCut> cut;
    std::vector<char> scr;
    if (batch_screen(b, p, cut, scr) && std::count(scr.begin(), scr.end(), 1) == (long)scr.size())
        dims &= ~(EPI_TUNE_ROWS | EPI_TUNE_QUEUES);
    epi_schedule cur = b->sched[form];
    double tcur = 0.0;
    int n = 0;
    rc = tune_descent(form, dims, cur, tcur, n, log, log_cap, [&](const epi_schedule &s, double &ms) -> int {
        b->sched[form] = s;
        int r = batch_prepare(b, p);
        if (r) return r;
        if ((r = batch_run(b, nullptr))) return r;  // warm-up
        std::vector<double> t(reps);
        for (int i = 0; i < reps; i++)
            if ((r = batch_run(b, &t[i]))) return r;
        std::sort(t.begin(), t.end());
        ms = t[reps / 2];
        return EPI_OK;
    });
    if (rc) return rc;
    b->sched[form] = cur;
    if (best) *best = cur;
    if (best_ms) *best_ms = tcur;
    if (nlog) *nlog = n;
    return EPI_OK;
}

int epi_batch_hit_count(epi_batch *b, int32_t scan, int64_t *nhits, int32_t *overflow)
{
    if (!b) return EPI_ERR_ARG;
    epi_ctx *c = b->ctx;
    if (scan < -1 || scan >= (int)b->scans.size()) return fail(c, EPI_ERR_ARG, "no such scan");
    if (overflow) *overflow = b->last_nhits > b->cap;
    if (scan < 0) {
        if (nhits) *nhits = b->last_nhits;
        return EPI_OK;
    }
    HIPCHK(c, hipSetDevice(c->device));
    int rc = batch_fetch(b);
    if (rc) return rc;
    if (nhits) *nhits = (int64_t)b->by_scan[scan].size();
    return EPI_OK;
}

int epi_batch_get_hits(epi_batch *b, int32_t scan, epi_hit *hits, double *F64, double *F2_64, int32_t *block,
                       int64_t cap, int64_t *n)
{
    if (!b || cap < 0) return EPI_ERR_ARG;
    epi_ctx *c = b->ctx;
    if (scan < 0 || scan >= (int)b->scans.size()) return fail(c, EPI_ERR_ARG, "no such scan");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = batch_fetch(b);
    if (rc) return rc;
    long long m = 0;
    emit_hits(*b->data[b->scans[scan].first], b->hh.data(), b->by_scan[scan], hits, F64, F2_64, block, cap, &m);
    if (n) *n = m;
    return EPI_OK;
}

int epi_batch_stats(epi_batch *b, double *kernel_ms, int64_t *pairs, int64_t *tiles, int32_t *captures,
                    int32_t *grid)
{
    if (!b) return EPI_ERR_ARG;
    if (grid) *grid = b->grid;
    if (kernel_ms) *kernel_ms = b->last_ms;
    if (pairs) *pairs = b->pairs;
    if (tiles) *tiles = b->nwork;
    if (captures) *captures = b->captures;
    return EPI_OK;
}

int epi_batch_last_screen(epi_batch *b, int32_t *scans, int64_t *candidates, int64_t *redone)
{
    if (!b) return EPI_ERR_ARG;
    if (scans) *scans = b->last_screened;
    if (candidates) *candidates = b->last_cand;
    if (redone) *redone = b->last_redone;
    return EPI_OK;
}

}  // extern "C"
