"""Which kernels a screened scan runs: batches of small and of large cohorts (tiles of 32 and of 64 rows) with FAST,
SPARSE and GENERAL lists, a scan that is not screened among them and strong SNPs whose regions exact tiles redo, and
a scan in pieces that has regions to redo. The counters of the screen show that the path was taken, and the
hits are those of the exact tiles (epi_scan_noalloc), bit for bit: both compute them from the same integers."""
import numpy as np
import pytest

import epigpu_amd as E
from epigpu_amd import scan as S
from test_gpu_screened import CAP, buf, phenotype, sch  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


def load(s, words, nid, y, sizes):
    s.set_genotypes(words, nid)
    s.set_phenotypes(y)
    s.set_chromosomes(list(np.cumsum([0] + sizes[:-1])), sizes)


def same_as_exact(s, buf, g, **kw):
    """The hits g of a screened scan against the exact tiles of the dataset in s."""
    n = s.scan_noalloc(buf.ptr.value, CAP, form="mfma", **kw)
    assert g["nhits"] == n <= CAP
    h = buf.read(S.HIT64_DTYPE, n)
    h = h[np.lexsort((h["snp2"], h["snp1"]))]
    o = np.lexsort((g["hits"]["snp2"], g["hits"]["snp1"]))
    for k in ("snp1", "snp2", "df1", "df2"):
        assert np.array_equal(h[k], g["hits"][k][o]), k
    assert np.array_equal(h["F"], g["F64"][o]) and np.array_equal(h["F2"], g["F2_64"][o])
    return n


def tiles(sizes, rows, cols):
    """Tiles of rows x cols over all chromosome pairs that hold a pair a > b."""
    start = np.cumsum([0] + sizes[:-1])
    n = 0
    for i in range(len(sizes)):
        for j in range(i + 1):
            for a in range(0, sizes[i], rows):
                a1 = start[i] + min(sizes[i], a + rows)
                n += sum(a1 - 1 > start[j] + b for b in range(0, sizes[j], cols))
    return n


@pytest.mark.parametrize("top,rows", [(1900, 32), (2100, 64)])
def test_batch_kernels(scanner, buf, top, rows):
    """The tile height follows the largest cohort; every list is screened, and has regions to redo."""
    data = [(900, [1300, 200], 0.0, 3), (1300, [901], 0.001, 2), (700, [500, 451], 0.02, 2), (top, [401], 0.0, 1)]
    t1, t2 = 4.5, 6.5
    with E.Batch(scanner) as b:
        made = []
        for i, (nid, sizes, gmiss, nphen) in enumerate(data):
            words = E.synth_genotypes(300 + i, nid, sum(sizes), 0.05, 0.5, gmiss)
            y = np.stack([phenotype(k, nid, 400 + i) for k in ("normal", "gamma", "casecontrol")[:nphen]])
            if i == 0:
                y[1, 7] = 1e4  # an outlier: this scan is not screened
            y[-1] += 1.5 * (S.unpack(words[60:64], nid) % 3).sum(0)  # rows of hits
            y[:, 5::13] = np.nan
            d = b.add_dataset(words, nid, list(np.cumsum([0] + sizes[:-1])), sizes)
            made += [(words, nid, sizes, yy, s) for yy, s in zip(y, b.add_phenotypes(d, y))]
        for rep in range(2):
            st = b.scan(test="i", t1=t1, t2=t2)
            scr = b.last_screen()
            print(f"batch top={top} replay={rep} {st} {scr}", flush=True)
            assert scr["scans"] == len(made) - 1
            assert scr["candidates"] > 0 and scr["redone"] > 0
            for words, nid, sizes, y, s in made:
                load(scanner, words, nid, y, sizes)
                assert same_as_exact(scanner, buf, b.hits(s), test="i", t1=t1, t2=t2) > 0
        # the two complete datasets by themselves: the list has exactly the tiles of this height
    with E.Batch(scanner) as b:
        n = 0
        for (words, nid, sizes, y, _) in (made[0], made[-1]):
            b.add_phenotypes(b.add_dataset(words, nid, list(np.cumsum([0] + sizes[:-1])), sizes), y)
            n += tiles(sizes, rows, 64)
        assert b.scan(test="i", t1=t1, t2=t2)["tiles"] == n
        assert b.last_screen()["scans"] == 2


@pytest.mark.parametrize("gmiss", [0.0, 0.01])
def test_pieces_with_regions(sch, buf, gmiss):
    """A scan in pieces of the tile list, every piece with regions to redo, against the exact tiles."""
    nid, sizes = 1500, [1700, 331]
    words = E.synth_genotypes(41, nid, sum(sizes), 0.1, 0.5, gmiss)
    y = (phenotype("normal", nid, 42) + 0.5 * (S.unpack(words[:12], nid) % 3).sum(0)).astype(np.float32)
    load(sch, words, nid, y, sizes)
    kw = dict(test="i", t1=6.5, t2=10.5)
    one = sch.scan(**kw)
    whole = sch.last_screen()
    try:
        sch.set_max_tiles(300)
        g = sch.scan(**kw)
        scr = sch.last_screen()
        print(f"pieces gmiss={gmiss} whole {one['launches']} {whole} pieces {g['launches']} {scr}", flush=True)
        assert g["launches"] > 2 * one["launches"]
        assert scr == whole and scr["digits"] > 0 and scr["candidates"] > 0 and scr["redone"] > 4
        assert same_as_exact(sch, buf, g, **kw) == one["nhits"]
    finally:
        sch.set_max_tiles(1 << 25)


def test_not_screened_counts(sch):
    """A scan below the least work, and a plain scan, report no screen."""
    words = E.synth_genotypes(43, 500, 200, 0.1, 0.5, 0.0)
    load(sch, words, 500, phenotype("normal", 500, 44), [200])
    for form in ("mfma", "plain"):
        sch.scan(form=form, t1=3.0, t2=4.0)
        assert sch.last_screen() == {"digits": 0, "candidates": 0, "redone": 0}


@pytest.mark.parametrize("nphen,gmiss", [(1, 0.0), (1, 0.01), (3, 0.0)])
def test_many_candidates(scanner, buf, nphen, gmiss):
    """More candidates than the list holds at a rate that admits the screen: the list is resolved in between, and no region
    goes to the exact tiles."""
    nid, nsnp = 600, 41000 if nphen == 1 else 24000
    words = E.synth_genotypes(51, nid, nsnp, 0.1, 0.5, gmiss)
    y = np.stack([phenotype("normal", nid, 52 + i) for i in range(nphen)])
    kw = dict(test="f", t1=float(S.f_isf(1.3e-3, 8, nid - 9)), t2=10.5)
    load(scanner, words, nid, y, [nsnp])
    one = [scanner.scan(phen=r, **kw) for r in range(nphen)]
    scr = scanner.last_screen()
    if nphen > 1:
        with E.Batch(scanner) as b:
            b.add_phenotypes(b.add_dataset(words, nid), y)
            for rep in range(2):
                b.scan(**kw)
                scr = dict(b.last_screen(), digits=1)
                for r in range(nphen):
                    g = b.hits(r)
                    assert all(np.array_equal(g[k], one[r][k]) for k in ("hits", "F64", "F2_64", "block"))
    print(f"candidates nphen={nphen} gmiss={gmiss} hits {[g['nhits'] for g in one]} {scr}", flush=True)
    assert scr["digits"] and scr["candidates"] > (1 << 20)
    assert scr["redone"] == 0
    assert same_as_exact(scanner, buf, one[0], **kw) > 0


def stratified(nid, nsnp, spread, seed):
    """Two populations with allele frequencies that differ by `spread` SDs, and a phenotype that differs between them."""
    rng = np.random.default_rng(seed)
    pop = np.arange(nid) % 2
    f = np.clip(rng.uniform(0.2, 0.5, nsnp)[:, None] + (rng.standard_normal(nsnp) * spread)[:, None] * pop, 0.02, 0.98)
    codes = sum((rng.random((nsnp, nid), dtype=np.float32) < f).astype(np.int8) for _ in range(2))
    return codes, (pop + rng.standard_normal(nid)).astype(np.float32)


@pytest.mark.parametrize("gmiss", [0.0, 0.01])
@pytest.mark.parametrize("nid", [1000, 2000])
def test_dense_blocks(scanner, buf, nid, gmiss):
    """Hits all over, where the screen expected none: the exact tiles redo blocks of 32 rows, each once."""
    sizes = [2500, 433]
    codes, y = stratified(nid, sum(sizes), 0.15, nid)
    if gmiss:
        codes[np.random.default_rng(1).random(codes.shape) < gmiss] = 3
    load(scanner, S.pack(codes), nid, y, sizes)
    kw = dict(test="i", t1=6.5, t2=10.5)
    g = scanner.scan(**kw)
    scr = scanner.last_screen()
    blocks = tiles(sizes, 32, 32 if gmiss else 64)
    print(f"dense nid={nid} gmiss={gmiss} hits {g['nhits']} of {g['pairs']} {scr} blocks {blocks}", flush=True)
    assert scr["digits"] and blocks / 2 < scr["redone"] <= blocks
    assert same_as_exact(scanner, buf, g, **kw) > 0.2 * g["pairs"]


@pytest.mark.parametrize("gmiss,dense_missing", [(0.0, 0), (0.002, 0), (0.002, 2), (0.02, 0)])
def test_batch_mixed(scanner, buf, gmiss, dense_missing):
    """Scans that are not screened (an outlier) keep the exact kernels of their tiles, beside screened ones of the same and of
    other datasets."""
    data = [(1000, [1600], 0.0, [0]), (2500, [1900, 433], gmiss, [1, 0, 1])]
    kw = dict(test="i", t1=5.0, t2=7.0)
    with E.Batch(scanner) as b:
        b.set_schedule("mfma", dense_missing=dense_missing)
        made = []
        for i, (nid, sizes, gm, outlier) in enumerate(data):
            words = E.synth_genotypes(61 + i, nid, sum(sizes), 0.1, 0.5, gm)
            y = np.stack([phenotype("normal", nid, 70 + i + 5 * r) for r in range(len(outlier))])
            y[np.array(outlier) == 1, 11] = 1e4
            y[0] += 8.0 / np.sqrt(nid) * (S.unpack(words[40:41], nid)[0] % 3)
            d = b.add_dataset(words, nid, list(np.cumsum([0] + sizes[:-1])), sizes)
            made += [(words, nid, sizes, yy, s) for yy, s in zip(y, b.add_phenotypes(d, y))]
        for rep in range(3):
            b.scan(**kw)
            scr = b.last_screen()
            print(f"mixed gmiss={gmiss} dense_missing={dense_missing} replay={rep} {b.stats()} {scr}", flush=True)
            assert scr["scans"] == 2 and scr["redone"] == 0
        for words, nid, sizes, y, s in made:
            load(scanner, words, nid, y, sizes)
            assert same_as_exact(scanner, buf, b.hits(s), **kw) > 0


def test_autotune_leaves_what_it_cannot_measure(sch):
    """The tuner does not time values that a screened scan ignores, and keeps them as they were."""
    nid, nsnp = 1000, 2000
    words = E.synth_genotypes(111, nid, nsnp, 0.1, 0.5, 0.0)
    y = phenotype("normal", nid, 112)
    load(sch, words, nid, y, [nsnp])
    for rows in (32, 64):
        sch.set_schedule("mfma", fast_rows=rows, super_a=8, super_b=4)
        r = sch.autotune(test="i")
        assert sch.last_screen()["digits"]
        assert {x["fast_rows"] for x in r["log"]} == {rows} and len(r["log"]) > 2
        assert sch.schedule("mfma")["fast_rows"] == rows
        # not screened: both heights are measured
        assert {x["fast_rows"] for x in sch.autotune(test="f", t1=1.5)["log"]} == {32, 64}
    with E.Batch(sch) as b:
        d = b.add_dataset(words, nid)
        b.add_phenotypes(d, y)
        for queues in (8, 1):
            b.set_schedule("mfma", fast_rows=64, queues=queues)
            r = b.autotune(test="i")
            assert b.last_screen()["scans"] == 1
            assert {(x["fast_rows"], x["queues"]) for x in r["log"]} == {(64, queues)} and len(r["log"]) > 2
        r = b.autotune(test="f", t1=1.5)
        assert {x["queues"] for x in r["log"]} == {1, 8} and {x["fast_rows"] for x in r["log"]} == {32, 64}
