"""Screened tiles whose third mask is the missing calls (cohorts from 3000 individuals on, 64-row tiles) against the
exact tiles, single scans and a batch: cohorts on both sides of that line and of the 128-individual step, SNPs
without any call, SNPs with all of them, and absent phenotypes among the missing calls. No tolerance: hits, F and F2 are
computed from the same integers."""
import numpy as np
import pytest

import epigpu_amd as E
from epigpu_amd import scan as S
from test_gpu_screened import CAP, both, buf, phenotype, sch  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


def dataset(nid, nsnp, gmiss, seed):
    """Words with one SNP of no calls, one that misses half, and three complete ones; phenotype with an additive effect."""
    rng = np.random.default_rng(seed)
    codes = S.unpack(E.synth_genotypes(seed, nid, nsnp, 0.02, 0.5, gmiss), nid).astype(np.int64)
    codes[5] = 3
    codes[6, rng.random(nid) < 0.5] = 3
    codes[nsnp // 2: nsnp // 2 + 3] = rng.integers(0, 3, (3, nid))
    snp = codes[-9] % 3
    y = phenotype("normal", nid, seed) + (9.0 / np.sqrt(nid) * (snp - snp.mean()) / snp.std()).astype(np.float32)
    y[3::17] = np.nan
    y[-1] = np.nan
    return S.pack(codes), y


@pytest.mark.parametrize("gmiss", [0.004, 0.08])
@pytest.mark.parametrize("nid,sizes", [(2944, [500, 130]), (2945, [500, 130]), (3001, [321, 65, 64]), (4096, [350]),
                                       (4225, [257, 63])])
def test_nocall(sch, buf, nid, sizes, gmiss):
    words, y = dataset(nid, sum(sizes), gmiss, nid)
    for test, p in (("i", 1e-4), ("f", 1e-4)):
        t1, t2 = (float(S.f_isf(p, d, nid - 9)) for d in (8, 4))
        print(f"nocall nid={nid} sizes={sizes} gmiss={gmiss} test={test}", flush=True)
        assert both(sch, buf, words, nid, y, sizes, test=test, t1=t1, t2=t2) > 0


def test_nocall_batch(scanner, buf):
    """One batch of cohorts on both sides of the line, one and two digits."""
    t1, t2 = 6.0, 8.0
    with E.Batch(scanner) as b:
        made = []
        for nid, nsnp, gmiss in ((2000, 400, 0.02), (3500, 300, 0.01), (20000, 150, 0.02)):
            words, y = dataset(nid, nsnp, gmiss, nid)
            y = np.stack([y, phenotype("gamma", nid, nid + 1)])
            d = b.add_dataset(words, nid)
            made += [(words, nid, nsnp, yy, s) for yy, s in zip(y, b.add_phenotypes(d, y))]
        for test in ("i", "f"):
            b.scan(test=test, t1=t1, t2=t2)
            for words, nid, nsnp, y, s in made:
                print(f"nocall batch test={test} nid={nid} scan={s}", flush=True)
                g = b.hits(s)
                scanner.set_genotypes(words, nid)
                scanner.set_phenotypes(y)
                scanner.set_chromosomes([0], [nsnp])
                n = scanner.scan_noalloc(buf.ptr.value, CAP, test=test, t1=t1, t2=t2)
                assert g["nhits"] == n
                h = buf.read(S.HIT64_DTYPE, n)
                h = h[np.lexsort((h["snp2"], h["snp1"]))]
                o = np.lexsort((g["hits"]["snp2"], g["hits"]["snp1"]))
                for k in ("snp1", "snp2", "df1", "df2"):
                    assert np.array_equal(h[k], g["hits"][k][o]), k
                assert np.array_equal(h["F"], g["F64"][o]) and np.array_equal(h["F2"], g["F2_64"][o])
