"""Plain-form tiles at the edges of their tiles (16 or 32 x 64 SNPs), words (32 individuals) and stages, against the
FP64 oracle: both tile heights, with and without missing calls, and phenotypes that span many powers of two.

Counts are exact. A cell's sum is made of at most nine accumulated sums (the four of its planes and their totals, by
subtraction). An accumulated sum adds up to 32 FP32 values by FMAs, so its error is at most 33 roundings (those of the
additions and of the value itself) of 2^-24 times the sum of |y - centre|, which is at most twice that of |y|; the
dump and the oracle's comparison add one rounding of the result. Hence 9 * 33 * 2^-24 * 2 * sum |y| + 2^-23 |sum|.
"""
import numpy as np
import pytest

import oracle as O
from conftest import make_dataset

pytestmark = pytest.mark.gpu


@pytest.fixture
def plain(scanner):
    saved = scanner.schedule("plain")
    yield scanner
    scanner.set_schedule("plain", **saved)


@pytest.mark.parametrize("gmiss", [0.0, 0.03])
@pytest.mark.parametrize("rows", [16, 32])
@pytest.mark.parametrize("nid,nsnp", [(6, 2), (31, 16), (32, 17), (33, 33), (64, 63), (65, 64), (255, 65), (256, 97),
                                      (257, 130), (1023, 31)])
def test_edges(plain, nid, nsnp, rows, gmiss):
    words, y = make_dataset(nid * 7 + nsnp, nid, nsnp, gmiss=gmiss, pmiss=0.05)
    for spread in (0, 12):
        # with a spread, every third value is up to 2^-60 of the others
        z = y.copy()
        if spread:
            z[::3] *= np.exp2(-5.0 * (np.arange(len(z[::3])) % (spread + 1))).astype(np.float32)
        print(f"plain {nid} x {nsnp} rows {rows} missing {gmiss} spread {spread}", flush=True)
        plain.set_genotypes(words, nid)
        plain.set_phenotypes(z)
        plain.set_schedule("plain", fast_rows=rows)
        counts, sums, _, _ = plain.pair_dump(0, nsnp, 0, nsnp, test="i", form="plain")
        aa, bb = np.meshgrid(np.arange(nsnp), np.arange(nsnp), indexing="ij")
        sel = aa > bb
        ref = O.pairs(O.unpack(words, nid), z, np.stack([aa[sel], bb[sel]], axis=1))
        assert (counts[sel] == ref["counts"]).all()
        tol = 9 * 33 * 2.0**-24 * 2 * np.nansum(np.abs(z)) + 2.0**-23 * np.abs(ref["sums"])
        assert (np.abs(sums[sel] - ref["sums"]) <= tol).all()
