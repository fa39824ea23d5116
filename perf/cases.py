"""Workloads of the pair scan, as a program that uses epigpu_amd runs them.

A case is a dict of plain values:
  kind    "scan"   one scan of genotypes and phenotypes that are already on the GPU (a study scanned
                   again with another phenotype, permutation or threshold): Scanner.scan
          "load"   a new study: genotypes, phenotype and chromosomes from host memory, then the scan
          "batch"  several scans in one call, every dataset with one or more phenotypes: Batch.scan
                   and the hits of each scan
  nid     individuals (kind "batch": of the largest dataset)
  nsnp    SNPs (likewise)
  nchr    chromosomes
  miss    mean rate of missing genotype calls
  ymiss   rate of missing phenotype values (NaN)
  maf     lowest minor allele frequency (the highest is 0.5)
  phen    distribution of the phenotype: normal, gamma, t5, binary (a case in four)
  test    "f" (8 df) or "i" (8 df and 4 df interaction)
  pval    0: the default thresholds 6.5 and 10.5; otherwise hits are pairs with p below it
  form    "mfma", or "plain", the independent form that cross-checks it
  safe    the reference's safe mode (-9 is a value, no condition on the number of cells)
  ndata, nphen   kind "batch": datasets, and phenotypes of each
  keep    rows of the table into which the program copies a scan's hits, in their order
Genotypes come in blocks of SNPs in linkage disequilibrium, with either allele counted; three pairs of
SNPs and one single SNP carry an effect on the phenotype.
"""
import math

import numpy as np
import torch

import epigpu_amd as E

BASE = dict(kind="scan", nid=1000, nsnp=1000, nchr=1, miss=0.0, ymiss=0.0, maf=0.05, phen="normal", test="i",
            pval=0.0, form="mfma", safe=False, ndata=1, nphen=1, keep=4096)

# Cost of one pair and individual relative to the others, to bound drawn cases.
UNIT = {("mfma", False): 16.0, ("mfma", True): 40.0, ("plain", False): 230.0, ("plain", True): 460.0}


def _case(name, **kw):
    c = dict(BASE, name=name)
    c.update(kw)
    return c


def listed():
    return [
        # A candidate-gene panel in a small cohort, 8 df test at a p-value: the smallest call, where
        # launches and the host's share count.
        _case("panel", nid=500, nsnp=2000, test="f", pval=1e-4, keep=1024),
        # A small study with ragged sizes on five chromosomes, missing calls and phenotypes.
        _case("ragged", nid=1237, nsnp=5003, nchr=5, miss=0.02, ymiss=0.03, maf=0.01),
        # A cohort of ordinary size with 1 % missing calls on two chromosomes.
        _case("cohort_missing", nid=4000, nsnp=20000, nchr=2, miss=0.01, ymiss=0.02, maf=0.01),
        # The same after quality control by call rate.
        _case("cohort_qc", nid=4000, nsnp=20000, nchr=2, miss=0.0025, ymiss=0.02, maf=0.01),
        # The benchmark's shape: imputed genotypes, a skewed quantitative trait; the largest case.
        _case("cohort_complete", nid=8000, nsnp=50000, phen="gamma", keep=32768),
        # A scan that keeps suggestive pairs (p < 1e-4): many hits to decide, collect and sort.
        _case("suggestive", nid=3001, nsnp=12007, nchr=3, pval=1e-4, phen="t5", keep=32768),
        # A large cohort over a candidate region, safe mode.
        _case("biobank", nid=50000, nsnp=4001, safe=True, phen="binary", pval=1e-6),
        # A new study from host memory: upload, transcode, phenotype preparation, scan.
        _case("new_study", kind="load", nid=2000, nsnp=20001, nchr=4, ymiss=0.01),
        # Sixteen independent small studies in one call.
        _case("studies", kind="batch", nid=6000, nsnp=12000, nchr=3, ymiss=0.03, ndata=16, keep=256),
        # Four traits of one large cohort with missing calls.
        _case("traits", kind="batch", nid=20000, nsnp=10000, miss=0.01, maf=0.01, nphen=4, phen="gamma"),
        # A permutation run: one complete study, sixteen phenotype vectors, 8 df test.
        _case("permutations", kind="batch", nid=2504, nsnp=8000, nchr=2, nphen=16, test="f"),
        # The plain form, as the cross-check of a study's result.
        _case("crosscheck", nid=1500, nsnp=6000, nchr=2, phen="gamma", form="plain"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sizes(case):
    """(nid, nsnp) of each dataset: the listed size, then sizes down to a twentieth of it (a tenth in SNPs)."""
    out = []
    for d in range(case["ndata"]):
        f = (0.6180339887 * d) % 1.0
        g = (0.7548776662 * d) % 1.0
        out.append((max(500, int(case["nid"] * (1 - 0.95 * f))), int(case["nsnp"] * (1 - 0.9 * g))))
    return out


def _cost(case):
    u = UNIT[case["form"], case["miss"] > 0]
    return sum(m * (m - 1) / 2 * n for n, m in _sizes(case)) * u * case["nphen"]


def draw(rng):
    limit = max(_cost(c) for c in listed())
    kind = rng.choice(["scan", "scan", "scan", "load", "batch"])
    c = dict(BASE, kind=kind)
    c["miss"] = rng.choice([0.0, 0.0, rng.uniform(0.0005, 0.005), rng.uniform(0.005, 0.03)])
    c["ymiss"] = rng.choice([0.0, rng.uniform(0.0, 0.1)])
    c["maf"] = rng.choice([0.01, 0.05])
    c["form"] = rng.choice(["mfma"] * 6 + ["plain"])
    c["phen"] = rng.choice(["normal", "gamma", "t5", "binary"])
    c["test"] = rng.choice("fii")
    c["pval"] = rng.choice([0.0, 0.0, 1e-4, 1e-6])
    c["safe"] = rng.random() < 0.15
    if kind == "batch":
        c["ndata"], c["nphen"] = rng.choice([(1, rng.randint(2, 12)), (rng.randint(2, 16), 1), (3, 2)])
    # tables with few cells, which rare alleles give, are hits by themselves without the condition on the cells
    if c["test"] == "f" or c["safe"]:
        c["maf"] = 0.05
    c["nid"] = _log(rng, 500, 40000)
    c["nsnp"] = _log(rng, 1000, 50000)
    while _cost(c) > limit:
        c["nsnp"] = max(1000, int(c["nsnp"] * 0.8))
        if c["nsnp"] == 1000:
            c["nid"] = max(500, int(c["nid"] * 0.8))
    c["keep"] = 256 if kind == "batch" else 32768 if c["pval"] == 1e-4 else 4096
    c["nchr"] = rng.randint(1, 6)
    return c


def _chromosomes(nsnp, nchr):
    """Uneven chromosome sizes that add up to nsnp."""
    w = [1.0 / (1.0 + 0.45 * i) for i in range(nchr)]
    cuts = [int(nsnp * sum(w[:i]) / sum(w)) for i in range(nchr)] + [nsnp]
    return cuts[:-1], [cuts[i + 1] - cuts[i] for i in range(nchr)]


def _thresholds(case, nid):
    """(t1, t2) of the tests F(8, nid - 9) and F(4, nid - 9)."""
    if not case["pval"]:
        return 6.5, 10.5

    def isf(p, d1, d2):
        # the F tail by Simpson's rule in v = 1 / (1 + x d1 / d2), bisected in log v
        def sf(x):
            v = d2 / (d2 + d1 * x)
            a, b = d2 / 2.0, d1 / 2.0
            lb = math.lgamma(a) + math.lgamma(b) - math.lgamma(a + b)
            t = np.linspace(-80.0 / a, 0.0, 4001)
            u = v * np.exp(t)
            y = np.exp(a * np.log(u) + (b - 1) * np.log1p(-u) - lb)
            w = np.full(t.size, 2.0)
            w[1::2] = 4.0
            w[0] = w[-1] = 1.0
            return float((y * w).sum() * (t[1] - t[0]) / 3.0)
        lo, hi = 1.0, 100.0
        for _ in range(60):
            mid = 0.5 * (lo + hi)
            lo, hi = (mid, hi) if sf(mid) > p else (lo, mid)
        return float(np.float32(0.5 * (lo + hi)))

    return isf(case["pval"], 8, nid - 9), isf(case["pval"], 4, nid - 9)


def _codes(case, nid, nsnp, seed):
    """(nsnp, nid) uint8 genotype codes on the GPU: 0, 1, 2 copies of the counted allele, 3 no call.

    Blocks of 8 SNPs share a latent uniform per haplotype, which each SNP takes with probability 0.8."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = torch.empty((nsnp, nid), dtype=torch.uint8, device="cuda")
    step = max(8, int(4e7 / nid) // 8 * 8)
    for s0 in range(0, nsnp, step):
        m = min(step, nsnp - s0)
        mb = (m + 7) // 8 * 8
        f = case["maf"] + (0.5 - case["maf"]) * torch.rand((mb, 1), generator=g, device="cuda")
        cnt = torch.zeros((mb, nid), dtype=torch.uint8, device="cuda")
        for _ in range(2):
            own = torch.rand((mb, nid), generator=g, device="cuda")
            shared = torch.rand((mb // 8, 1, nid), generator=g, device="cuda").expand(-1, 8, -1).reshape(mb, nid)
            pick = torch.rand((mb, nid), generator=g, device="cuda") < 0.8
            cnt += (torch.where(pick, shared, own) < f).to(torch.uint8)
        flip = torch.rand((mb, 1), generator=g, device="cuda") < 0.5
        cnt = torch.where(flip, 2 - cnt, cnt)
        if case["miss"]:
            rate = 2.0 * case["miss"] * torch.rand((mb, 1), generator=g, device="cuda")
            none = torch.rand((mb, nid), generator=g, device="cuda") < rate
            cnt = torch.where(none, torch.full_like(cnt, 3), cnt)
        out[s0:s0 + m] = cnt[:m]
    return out


def _phenotypes(case, codes, seed):
    """(nphen, nid) float32 phenotypes (NaN missing): three SNP pairs interact in heterozygotes without main
    effects, and one SNP has an additive effect of its own."""
    nsnp, nid = codes.shape
    rng = np.random.default_rng(seed)
    pairs = [rng.choice(nsnp, 2, replace=False) for _ in range(3)]
    rows = codes[torch.as_tensor(np.concatenate(pairs), device="cuda")].cpu().numpy()

    def unit(x):
        x = x - x.mean()
        return x / max(x.std(), 1e-3)

    het = [unit(r == 1) for r in rows]
    effect = sum(unit(het[2 * i] * het[2 * i + 1]) for i in range(3)) * (11.0 / math.sqrt(nid))
    effect += unit(np.where(rows[0] == 3, 1, rows[0]).astype(float)) * (5.0 / math.sqrt(nid))
    ys = []
    for _ in range(case["nphen"]):
        d = case["phen"]
        if d == "normal":
            y = rng.standard_normal(nid)
        elif d == "gamma":
            y = (rng.gamma(2.0, 1.0, nid) - 2.0) / math.sqrt(2.0)
        elif d == "t5":
            y = rng.standard_t(5, nid)
        else:
            y = rng.standard_normal(nid)
        y = y + effect
        if d == "binary":
            y = y > 0.6745
        y = y.astype(np.float32)
        if case["ymiss"]:
            y[rng.random(nid) < case["ymiss"]] = np.nan
        ys.append(y)
    return np.stack(ys)


def _pack(codes):
    """Packed words: 16 genotypes per int32, the first in the two highest bits; a shorter tail word is
    right-aligned."""
    nsnp, nid = codes.shape
    full, rem = nid // 16, nid % 16
    words = torch.zeros((nsnp, full + (rem > 0)), dtype=torch.int64, device="cuda")
    c = codes[:, :16 * full].reshape(nsnp, full, 16)
    for t in range(16):
        words[:, :full] |= c[:, :, t].to(torch.int64) << (30 - 2 * t)
    for t in range(rem):
        words[:, full] |= codes[:, 16 * full + t].to(torch.int64) << (2 * (rem - 1 - t))
    return words.to(torch.int32).cpu().numpy()


def _datasets(case, seed):
    for d, (nid, nsnp) in enumerate(_sizes(case)):
        codes = _codes(case, nid, nsnp, 1000003 * seed + 7919 * d + 1)
        yield codes, _phenotypes(case, codes, [seed, d])


def prepare(case, seed):
    data = [(_pack(codes), y, codes.shape[1], _chromosomes(codes.shape[0], case["nchr"]))
            for codes, y in _datasets(case, seed)]
    t1, t2 = _thresholds(case, case["nid"])
    st = {"case": case, "args": dict(test=case["test"], form=case["form"], t1=t1, t2=t2, safe=case["safe"])}
    sc = st["scanner"] = E.Scanner(0)
    if case["kind"] == "batch":
        b = st["batch"] = E.Batch(sc)
        st["scans"] = []
        for words, y, nid, (start, size) in data:
            i = b.add_dataset(words, nid, start, size)
            st["scans"] += b.add_phenotypes(i, y, nine_is_value=case["safe"])
    elif case["kind"] == "load":
        st["data"] = data[0]
    else:
        _load(sc, data[0], case)
    return st


def _load(sc, data, case):
    words, y, nid, (start, size) = data
    sc.set_genotypes(words, nid)
    sc.set_phenotypes(y, nine_is_value=case["safe"])
    sc.set_chromosomes(start, size)


def _table(case, nhits, cols):
    """The hits' columns as a program keeps them: the first `keep` rows, zeros behind the last hit."""
    n = min(len(cols["snp1"]), case["keep"])
    out = {"nhits": nhits}
    for k, dtype in (("snp1", np.int32), ("snp2", np.int32), ("df1", np.int32), ("df2", np.int32),
                     ("block", np.int32), ("F", np.float32), ("F2", np.float32), ("F64", np.float64),
                     ("F2_64", np.float64)):
        t = out[k] = np.zeros(case["keep"], dtype)
        t[:n] = cols[k][:n]
    return out


def _join(tables):
    """One table of all scans."""
    return {k: np.stack([t[k] for t in tables]) for k in tables[0]}


def _hits(case, r):
    h = r["hits"]
    return _table(case, r["nhits"], dict(r, **{k: h[k] for k in h.dtype.names}))


def run(state):
    case, sc = state["case"], state["scanner"]
    if case["kind"] == "batch":
        b = state["batch"]
        b.scan(**state["args"])
        return _join([_hits(case, b.hits(s)) for s in state["scans"]])
    if case["kind"] == "load":
        _load(sc, state["data"], case)
    return _hits(case, sc.scan(**state["args"]))


def work(case):
    """Genotypes (2 bits) and phenotypes read once. Per pair and individual a multiply-add for the count and
    one for the sum of each independent cell (four without missing calls, the others following from the
    SNPs' own counts and sums; nine with them, and one more for the sum of squares)."""
    byts = flops = 0.0
    for nid, nsnp in _sizes(case):
        byts += nid * nsnp / 4 + 4.0 * nid * case["nphen"]
        per = 2 * (9 * 2 + 1) if case["miss"] else 2 * (4 * 2)
        flops += nsnp * (nsnp - 1) / 2 * nid * per * case["nphen"]
    return {"bytes": byts, "flops": flops}


def _exact_scan(case, codes, y, start, size, t1, t2):
    """Hits of one scan from FP64 products of the class indicators; None if a pair lies on a threshold."""
    nsnp, nid = codes.shape
    yt = torch.as_tensor(y, device="cuda", dtype=torch.float64)
    v = ~torch.isnan(yt)
    if not case["safe"]:
        v &= yt != -9.0
    keep = torch.nonzero(v)[:, 0]
    yt = yt[keep] - yt[keep].mean()
    codes = codes[:, keep]
    step = 4096
    hits = []

    def masks(lo, hi):
        return [(codes[lo:hi] == g) for g in range(3)]

    for i in range(len(start)):
        for j in range(i + 1):
            for a0 in range(start[i], start[i] + size[i], step):
                a1 = min(a0 + step, start[i] + size[i])
                A = masks(a0, a1)
                for b0 in range(start[j], start[j] + size[j], step):
                    b1 = min(b0 + step, start[j] + size[j])
                    if a1 - 1 <= b0:
                        continue
                    B = masks(b0, b1)
                    n, s = [], []
                    for g in range(3):
                        Ay = A[g].double() * yt
                        Af = A[g].float()
                        for h in range(3):
                            n.append((Af @ B[h].float().T).double())
                            s.append(Ay @ B[h].double().T)
                    if case["miss"]:
                        sq = ((codes[a0:a1] != 3).double() * (yt * yt)) @ (codes[b0:b1] != 3).double().T
                    else:
                        sq = (yt * yt).sum()
                    N, T = sum(n), sum(s)
                    nfac = sum((x > 0).double() for x in n)
                    mean = T / N
                    m = [torch.where(x > 0, z / x.clamp(min=1), torch.zeros_like(z)) for x, z in zip(n, s)]
                    ssb = sum(x * (z - mean) ** 2 for x, z in zip(n, m))
                    d1, d2 = nfac - 1, N - nfac
                    msw = (sq - N * mean * mean - ssb) / d2
                    F = ssb / d1 / msw
                    near = (F / t1 - 1).abs() < 3e-7
                    hit = F > t1
                    F2 = torch.zeros_like(F)
                    if case["test"] == "i":
                        R = [sum(s[3 * g:3 * g + 3]) / sum(n[3 * g:3 * g + 3]).clamp(min=1) for g in range(3)]
                        C = [sum(s[h::3]) / sum(n[h::3]).clamp(min=1) for h in range(3)]
                        ssi = sum(n[c] * (m[c] - R[c // 3] - C[c % 3] + mean) ** 2 for c in range(9))
                        F2 = ssi / 4 / msw
                        near |= (F2 / t2 - 1).abs() < 3e-7
                        hit |= F2 > t2
                        if not case["safe"]:
                            hit &= nfac > 6
                    ok = (d1 >= 1) & (d2 >= 1)
                    ai = torch.arange(a0, a1, device="cuda")[:, None]
                    bi = torch.arange(b0, b1, device="cuda")[None, :]
                    ok &= ai > bi
                    if bool((near & ok).any()):
                        return None
                    w = torch.nonzero(hit & ok)
                    if len(w):
                        r, c = w[:, 0], w[:, 1]
                        hits.append(torch.stack([torch.full_like(r, i * (i + 1) // 2 + j).double(),
                                                 (a0 + r).double(), (b0 + c).double(), d1[r, c], d2[r, c], F[r, c],
                                                 F2[r, c]], 1).cpu().numpy())
    h = np.concatenate(hits) if hits else np.zeros((0, 7))
    h = h[np.lexsort((h[:, 2], h[:, 1], h[:, 0]))]
    return _table(case, len(h), dict(snp1=h[:, 1], snp2=h[:, 2], df1=h[:, 3], df2=h[:, 4], block=h[:, 0],
                                     F=h[:, 5], F2=h[:, 6], F64=h[:, 5], F2_64=h[:, 6]))


def exact(case, seed):
    # about 18 products of every block of pairs in 64 bits: a few seconds at this bound
    if sum(m * m * n for n, m in _sizes(case)) * (1 + case["nphen"]) > 5e13:
        return None
    t1, t2 = _thresholds(case, case["nid"])
    out = []
    for codes, ys in _datasets(case, seed):
        start, size = _chromosomes(codes.shape[0], case["nchr"])
        for y in ys:
            r = _exact_scan(case, codes, y, start, size, t1, t2)
            if r is None:
                return None
            out.append(r)
    return _join(out) if case["kind"] == "batch" else out[0]
