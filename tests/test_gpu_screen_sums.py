"""The sums that the screen takes its bounds from, against integers: counts and sums of the coarse phenotype of every
cell, exact in FP32 MFMA accumulators as long as they stay below 2^24 units of 1/64. The sizes lie around the 128-individual
stage, the 16,384-individual window of weights, both tile heights and the line from which missing calls are contracted;
the phenotypes reach the largest sums there are (skewed, and sorted, so that partial sums grow before they cancel). No tolerance."""
import numpy as np
import pytest

import epigpu_amd as E
from epigpu_amd import scan as S
from test_gpu_screened import phenotype

pytestmark = pytest.mark.gpu


def expected(codes, v, present, a, b):
    """Counts and sums of v per cell of SNPs a x b, int64."""
    ca, cb = codes[a], codes[b]
    n = np.zeros((len(ca), len(cb), 9), dtype=np.int64)
    s = np.zeros_like(n)
    for g in range(3):
        ma = ((ca == g) & present).astype(np.float64)
        for h in range(3):
            mb = (cb == h).astype(np.float64)
            n[:, :, 3 * g + h] = np.rint(ma @ mb.T)
            s[:, :, 3 * g + h] = np.rint((ma * v) @ mb.T)
    return n, s


@pytest.mark.parametrize("kind", ["normal", "lognormal", "casecontrol", "ordered"])
@pytest.mark.parametrize("gmiss", [0.0, 0.05])
@pytest.mark.parametrize("nid", [100, 129, 1999, 2000, 2945, 3201, 16385, 33000, 65000])
def test_sums_are_exact(scanner, nid, gmiss, kind):
    nsnp = 150
    words = E.synth_genotypes(nid, nid, nsnp, 0.02, 0.5, gmiss)
    codes = S.unpack(words, nid)
    y = phenotype(kind, nid, nid + 1)
    if kind in ("casecontrol", "ordered"):
        codes[9] = 1  # a SNP that all share: its cells hold the whole sums
        codes[140] = np.where(np.arange(nid) < nid // 2, 0, 2)
        words = S.pack(codes)
    y[3::17] = np.nan
    scanner.set_genotypes(words, nid)
    scanner.set_phenotypes(y)
    a, b = np.arange(70, 150), np.arange(0, 100)
    below = a[:, None] > b[None, :]
    for digits in (1, 2):
        v, n, s = scanner.screen_dump(digits, 70, 150, 0, 100)
        present = ~np.isnan(y)
        assert (v[~present] == 0).all() and np.abs(v).max() <= (60 if digits == 1 else 1980)
        assert np.abs(v).sum() < 1 << 24
        want_n, want_s = expected(codes, v.astype(np.float64), present, a, b)
        print(f"sums nid={nid} gmiss={gmiss} {kind} digits={digits} largest {np.abs(want_s).max()}", flush=True)
        assert np.array_equal(64.0 * n[below], want_n[below])
        assert np.array_equal(64.0 * s[below], want_s[below])
        assert np.isnan(n[~below]).all() and np.isnan(s[~below]).all()


def test_sums_of_a_large_cohort(scanner):
    """300,000 individuals: one digit alone is coarse enough for its sums to stay exact."""
    nid, nsnp = 300000, 40
    words = E.synth_genotypes(7, nid, nsnp, 0.1, 0.5, 0.02)
    codes = S.unpack(words, nid)
    for kind in ("normal", "casecontrol"):
        y = phenotype(kind, nid, 8)
        scanner.set_genotypes(words, nid)
        scanner.set_phenotypes(y)
        v, n, s = scanner.screen_dump(1, 0, nsnp, 0, nsnp)
        assert 0 < np.abs(v).sum() < 1 << 24
        want_n, want_s = expected(codes, v.astype(np.float64), np.ones(nid, bool), np.arange(nsnp), np.arange(nsnp))
        below = np.tril(np.ones((nsnp, nsnp), bool), -1)
        print(f"sums nid={nid} {kind} largest {np.abs(want_s).max()}", flush=True)
        assert np.array_equal(64.0 * n[below], want_n[below]) and np.array_equal(64.0 * s[below], want_s[below])
        if kind == "normal":
            with pytest.raises(E.EpiError):
                scanner.screen_dump(2, 0, nsnp, 0, nsnp)
