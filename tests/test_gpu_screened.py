"""Screened scans (6-bit contraction and bound, exact resolve of the candidates) against the exact tiles.

epi_scan_noalloc runs the exact tiles on the same context, so its records are the reference: epi_scan must find the
same pairs with bit-identical F and F2. The sizes are those at which the screen can go wrong: cohorts around the
128-individual stage, the 256-individual padding and the 16,384-individual window of weights, SNP counts and chromosomes
around the 16 x 64 region of a wave, regions with so many hits that the exact tile redoes them, more candidates
than the candidate list holds, phenotypes of every shape that the fixed point takes, ordered cohorts (long partial
sums) and cells left empty by rare alleles. No tolerance: the values are computed from the same integers.
"""
import numpy as np
import pytest

import epigpu_amd as E
from epigpu_amd import scan as S
from test_zz_no_alloc import DevBuf

pytestmark = pytest.mark.gpu

CAP = 1 << 22


@pytest.fixture(scope="module")
def buf():
    b = DevBuf(CAP * S.HIT64_DTYPE.itemsize)
    yield b
    b.free()


@pytest.fixture
def sch(scanner):
    saved = scanner.schedule("mfma")
    yield scanner
    scanner.set_schedule("mfma", **saved)


def phenotype(kind, nid, seed):
    rng = np.random.default_rng(seed)
    y = {"normal": rng.standard_normal, "gamma": lambda n: rng.gamma(2.0, 1.0, n) + 50.0,
         "t5": lambda n: rng.standard_t(5, n), "lognormal": lambda n: np.exp(rng.standard_normal(n)),
         "binary": lambda n: (rng.random(n) < 0.3).astype(float),
         "ordered": lambda n: np.sort(rng.standard_normal(n)),
         "casecontrol": lambda n: (np.arange(n) < 0.4 * n).astype(float)}[kind](nid)
    return y.astype(np.float32)


def both(s, buf, words, nid, y, sizes, screened=True, **kw):
    """epi_scan and epi_scan_noalloc of one dataset; checks that they agree and returns the hit count."""
    s.set_genotypes(words, nid)
    s.set_phenotypes(y, nine_is_value=kw.get("safe", False))
    s.set_chromosomes(list(np.cumsum([0] + sizes[:-1])), sizes)
    g = s.scan(form="mfma", **kw)
    assert (g["launches"] > 1) == screened, g["launches"]
    n = s.scan_noalloc(buf.ptr.value, CAP, form="mfma", **kw)
    assert g["nhits"] == n <= CAP
    h = buf.read(S.HIT64_DTYPE, n)
    h = h[np.lexsort((h["snp2"], h["snp1"]))]
    o = np.lexsort((g["hits"]["snp2"], g["hits"]["snp1"]))
    for k in ("snp1", "snp2", "df1", "df2"):
        assert np.array_equal(h[k], g["hits"][k][o]), k
    assert np.array_equal(h["F"], g["F64"][o]) and np.array_equal(h["F2"], g["F2_64"][o])
    return n


@pytest.mark.parametrize("rows", [32, 64])
@pytest.mark.parametrize("nid,sizes", [(64, [4100]), (127, [2900, 17]), (128, [2881, 1, 63]), (129, [1500, 1401]),
                                       (500, [1025, 16, 15, 700]), (1025, [1100, 65]), (16384, [300]), (16385, [257, 31]),
                                       (33000, [191])])
def test_screened_sizes(sch, buf, rows, nid, sizes):
    seed = nid + rows
    nsnp = sum(sizes)
    words = E.synth_genotypes(seed, nid, nsnp, 0.02, 0.5, 0.0)
    sch.set_schedule("mfma", fast_rows=rows)
    t1, t2 = (float(S.f_isf(1e-5, d, nid - 9)) for d in (8, 4))
    snp = S.unpack(words[-9:-8], nid)[0].astype(float)  # an additive effect, so that some pairs are hits for certain
    effect = 8.0 / np.sqrt(nid) * (snp - snp.mean()) / snp.std()
    for test, safe in (("i", False), ("f", False), ("i", True)):
        print(f"screened rows={rows} nid={nid} sizes={sizes} test={test} safe={safe}", flush=True)
        y = phenotype("normal", nid, seed) + effect.astype(np.float32)
        y[3::17] = np.nan
        assert both(sch, buf, words, nid, y, sizes, test=test, safe=safe, t1=t1, t2=t2) > 0


@pytest.mark.parametrize("kind", ["gamma", "t5", "lognormal", "binary", "ordered", "casecontrol"])
def test_screened_phenotypes(sch, buf, kind):
    nid, sizes = 3000, [700, 500]
    words = E.synth_genotypes(77, nid, sum(sizes), 0.02, 0.5, 0.0)
    y = phenotype(kind, nid, 78)
    for p in (1e-4, 1e-6):
        t1, t2 = (float(S.f_isf(p, d, nid - 9)) for d in (8, 4))
        print(f"screened phenotype={kind} p={p}", flush=True)
        both(sch, buf, words, nid, y, sizes, test="i", t1=t1, t2=t2)
        both(sch, buf, words, nid, y, sizes, test="f", t1=t1, t2=t2)


@pytest.mark.parametrize("rows", [32, 64])
def test_screened_strong_snps(sch, buf, rows):
    """Four neighbouring SNPs with a strong main effect: all pairs of their rows are hits, so their regions go
    to the exact tile; a copy of one of them at every 16th SNP: more candidates than the list holds, while no region
    has enough for the exact tile."""
    nid, nsnp = 600, 5200
    words = E.synth_genotypes(5, nid, nsnp, 0.2, 0.5, 0.0)
    codes = S.unpack(words, nid)
    rng = np.random.default_rng(6)
    sch.set_schedule("mfma", fast_rows=rows)
    y = (codes[1000:1004].sum(0) + 0.5 * rng.standard_normal(nid)).astype(np.float32)
    assert both(sch, buf, words, nid, y, [nsnp], test="f", t1=6.5, t2=10.5) > 4 * nsnp * 0.9
    words2 = words.copy()
    words2[::16] = words[1000]
    y = (codes[1000] + rng.standard_normal(nid)).astype(np.float32)
    assert both(sch, buf, words2, nid, y, [nsnp], test="f", t1=6.5, t2=10.5) > (1 << 20)


@pytest.mark.parametrize("rows", [32, 64])
@pytest.mark.parametrize("gmiss", [0.002, 0.02, 0.1])
@pytest.mark.parametrize("nid,sizes", [(120, [2900, 17]), (129, [1500, 1401]), (500, [1025, 16, 15, 33]), (1025, [700, 65]),
                                       (16384, [300]), (16640, [257, 31])])
def test_screened_missing(sch, buf, rows, gmiss, nid, sizes):
    """GENERAL tiles, and at the lowest rate SPARSE ones among them."""
    seed = nid + rows
    words = E.synth_genotypes(seed, nid, sum(sizes), 0.02, 0.5, gmiss)
    sch.set_schedule("mfma", fast_rows=rows)
    t1, t2 = (float(S.f_isf(1e-5, d, nid - 9)) for d in (8, 4))
    snp = S.unpack(words[-9:-8], nid)[0].astype(float) % 3  # an additive effect (missing calls as class 0)
    effect = 9.0 / np.sqrt(nid) * (snp - snp.mean()) / snp.std()
    for test, safe, kind in (("i", False, "normal"), ("f", False, "casecontrol"), ("i", True, "gamma")):
        print(f"screened rows={rows} nid={nid} sizes={sizes} gmiss={gmiss} test={test} safe={safe}", flush=True)
        y = phenotype(kind, nid, seed) + effect.astype(np.float32)
        y[3::17] = np.nan
        assert both(sch, buf, words, nid, y, sizes, test=test, safe=safe, t1=t1, t2=t2) > 0
        kinds = sch.last_tiles()
        assert kinds["general"] + kinds["sparse"] > 0, kinds


@pytest.mark.parametrize("rows", [32, 64])
def test_screened_missing_strong_snps(sch, buf, rows):
    """Regions that the exact GENERAL tile redoes, and more candidates than the list holds, as without missing calls."""
    nid, nsnp = 600, 5200
    words = E.synth_genotypes(15, nid, nsnp, 0.2, 0.5, 0.01)
    codes = S.unpack(words, nid) % 3
    rng = np.random.default_rng(16)
    sch.set_schedule("mfma", fast_rows=rows)
    y = (codes[1000:1004].sum(0) + 0.5 * rng.standard_normal(nid)).astype(np.float32)
    assert both(sch, buf, words, nid, y, [nsnp], test="f", t1=6.5, t2=10.5) > 4 * nsnp * 0.9
    words2 = words.copy()
    words2[::16] = words[1000]
    y = (codes[1000] + rng.standard_normal(nid)).astype(np.float32)
    assert both(sch, buf, words2, nid, y, [nsnp], test="f", t1=6.5, t2=10.5) > (1 << 20)


@pytest.mark.parametrize("rows", [32, 64])
def test_screened_batch(scanner, buf, rows):
    """A batch over FAST, SPARSE and GENERAL lists, several phenotypes per dataset, one of them with outliers (its tiles
    are redone whole), one dataset of strong SNPs; every scan against the exact tiles, over three replays."""
    data = [(900, [1300, 200], 0.0, 3), (1300, [900], 0.001, 2), (700, [500, 450], 0.02, 2), (17000, [150], 0.0, 1)]
    t1, t2 = 4.5, 6.5
    with E.Batch(scanner) as b:
        b.set_schedule("mfma", fast_rows=rows)
        made = []
        for i, (nid, sizes, gmiss, nphen) in enumerate(data):
            words = E.synth_genotypes(100 + i, nid, sum(sizes), 0.05, 0.5, gmiss)
            y = np.stack([phenotype(k, nid, 200 + i) for k in ("normal", "gamma", "casecontrol")[:nphen]])
            if i == 0:
                y[1, 7] = 1e4  # an outlier
                y[2] += 1.5 * S.unpack(words[60:64], nid).sum(0)
            y[:, 5::13] = np.nan
            starts = list(np.cumsum([0] + sizes[:-1]))
            d = b.add_dataset(words, nid, starts, sizes)
            made += [(words, nid, sizes, yy, s) for yy, s in zip(y, b.add_phenotypes(d, y))]
        for rep in range(3):
            b.scan(test="i", t1=t1, t2=t2)
            for words, nid, sizes, y, s in made:
                print(f"screened batch rows={rows} replay={rep} scan={s}", flush=True)
                g = b.hits(s)
                scanner.set_genotypes(words, nid)
                scanner.set_phenotypes(y)
                scanner.set_chromosomes(list(np.cumsum([0] + sizes[:-1])), sizes)
                n = scanner.scan_noalloc(buf.ptr.value, CAP, test="i", t1=t1, t2=t2)
                assert g["nhits"] == n > 0
                h = buf.read(S.HIT64_DTYPE, n)
                h = h[np.lexsort((h["snp2"], h["snp1"]))]
                o = np.lexsort((g["hits"]["snp2"], g["hits"]["snp1"]))
                for k in ("snp1", "snp2", "df1", "df2"):
                    assert np.array_equal(h[k], g["hits"][k][o]), k
                assert np.array_equal(h["F"], g["F64"][o]) and np.array_equal(h["F2"], g["F2_64"][o])


def test_not_screened(sch, buf):
    """Thresholds that most pairs pass, negative ones, few pairs and phenotypes with outliers keep the exact tiles."""
    nid, nsnp = 800, 1400
    words = E.synth_genotypes(9, nid, nsnp, 0.05, 0.5, 0.0)
    y = phenotype("normal", nid, 10)
    assert both(sch, buf, words, nid, y, [nsnp], test="f", t1=6.5, t2=10.5) >= 0
    assert both(sch, buf, words, nid, y, [nsnp], screened=False, test="f", t1=1.5, t2=10.5) > 1000
    assert both(sch, buf, words, nid, y, [nsnp], screened=False, test="i", t1=6.5, t2=-1.0) > 1000
    assert both(sch, buf, words[:300], nid, y, [300], screened=False, test="f", t1=3.0, t2=10.5) > 0
    # so do datasets with many missing calls
    gone = E.synth_genotypes(9, nid, nsnp, 0.05, 0.5, 0.2)
    assert both(sch, buf, gone, nid, y, [nsnp], screened=False, test="f", t1=4.0, t2=10.5) > 0
    y[5] = 1e4
    both(sch, buf, words, nid, y, [nsnp], screened=False, test="f", t1=6.5, t2=10.5)
