"""Device memory of screened scans: what they can do without does not keep another dataset out.

The device is filled up to what two datasets take with their bitplanes alone (two copies, the class planes and the planes by
frequency) and the packed words of the second during its upload. The planes by SNP, which only make the resolve
kernel faster, fit for the first dataset by itself and have to be given back for the second. Afterwards both are
scanned, still screened, and their hits are those of scans with enough memory."""
import ctypes

import numpy as np
import pytest

import epigpu_amd as E
from test_gpu_screened import phenotype

pytestmark = pytest.mark.gpu

MIB = 1 << 20


class Hog:
    """Device memory taken until only `left` bytes are free."""

    def __init__(self, left):
        self.hip = ctypes.CDLL("libamdhip64.so.7")
        self.got = []
        for piece in (1 << 33, 1 << 30, 1 << 27, 1 << 24, 1 << 22):
            while self.free_bytes() >= left + piece:
                p = ctypes.c_void_p()
                if self.hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(piece)) != 0:
                    self.hip.hipGetLastError()
                    break
                self.got.append(p)

    def free_bytes(self):
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    def release(self):
        while self.got:
            self.hip.hipFree(self.got.pop())


def test_planes_by_snp_are_given_back():
    nid, nsnp, unit = 20000, 60000, 1500
    words = np.tile(E.synth_genotypes(91, nid, unit, 0.1, 0.5, 0.0), (nsnp // unit, 1))
    snp = E.unpack(words[7:8], nid)[0].astype(float)
    ys = [(phenotype("normal", nid, 92 + i) + 12.0 / np.sqrt(nid) * (snp - snp.mean()) / snp.std()).astype(np.float32)
          for i in range(2)]
    kw = dict(test="f", t1=9.0, t2=10.5)
    sizes = [1500, 500]  # what is scanned: the rest of the SNPs belongs to no chromosome
    starts = [0, 1500]
    plane = 3 * ((nid + 255) // 256 * 8) * nsnp * 4
    packed = words.nbytes
    with E.Scanner(0) as s:
        # every kernel has run once before the memory is short
        s.set_genotypes(words[:2000], nid)
        want = []
        for y in ys:
            s.set_phenotypes(y)
            s.set_chromosomes(starts, sizes)
            want.append(s.scan(**kw))
            assert s.last_screen()["digits"] and want[-1]["nhits"] > 0
        with E.Batch(s) as b:
            b.add_phenotypes(b.add_dataset(words[:2000], nid, starts, sizes), ys[0])
            b.scan(**kw)
        with E.Batch(s) as b:
            hog = Hog(4 * plane + packed + plane // 4)
            try:
                print(f"planes {plane / MIB:.0f} MiB, packed {packed / MIB:.0f}, free {hog.free_bytes() / MIB:.0f}", flush=True)
                scans = [b.add_phenotypes(b.add_dataset(words, nid, starts, sizes), y)[0] for y in ys]
                print(f"free with both datasets: {hog.free_bytes() / MIB:.0f} MiB", flush=True)
                for rep in range(2):
                    b.scan(**kw)
                    assert b.last_screen()["scans"] == 2 and b.last_screen()["candidates"] > 0
                    for scan, w in zip(scans, want):
                        g = b.hits(scan)
                        assert all(np.array_equal(g[k], w[k]) for k in ("hits", "F64", "F2_64", "block"))
            finally:
                hog.release()


@pytest.mark.parametrize("gmiss", [0.0, 0.02])
def test_candidates_from_the_bitplanes(gmiss):
    """Scans whose planes by SNP were given back find the same hits: a context keeps them until an allocation fails."""
    nid, sizes = 3001, [900, 801]
    words = E.synth_genotypes(95, nid, sum(sizes), 0.05, 0.5, gmiss)
    y = phenotype("gamma", nid, 96)
    kw = dict(test="i", t1=float(E.f_isf(1e-4, 8, nid - 9)), t2=float(E.f_isf(1e-4, 4, nid - 9)))
    with E.Scanner(0) as s:
        s.set_genotypes(words, nid)
        s.set_phenotypes(y)
        s.set_chromosomes([0, sizes[0]], sizes)
        a = s.scan(**kw)
        with pytest.raises(E.EpiError):
            s.set_hit_capacity(1 << 40)  # more than the card holds: the planes are given back, and it fails all the same
        s.set_hit_capacity(1 << 22)
        b = s.scan(**kw)
        assert s.last_screen()["digits"] and s.last_screen()["candidates"] > 0
        assert a["nhits"] == b["nhits"] > 0
        assert all(np.array_equal(a[k], b[k]) for k in ("hits", "F64", "F2_64", "block"))


def test_failed_hit_capacity():
    """A hit buffer that cannot be had: scans count their hits, store none and report the overflow; a later one serves again."""
    nid, nsnp = 700, 1500
    words = E.synth_genotypes(97, nid, nsnp, 0.1, 0.5, 0.0)
    y = phenotype("normal", nid, 98)
    kw = dict(test="f", t1=3.5, t2=10.5)
    with E.Scanner(0) as s, E.Batch(s) as b:
        s.set_genotypes(words, nid)
        s.set_phenotypes(y)
        b.add_phenotypes(b.add_dataset(words, nid), y)
        want = s.scan(**kw)
        b.scan(**kw)
        assert b.hits(0)["nhits"] == want["nhits"] > 0
        for x in (s, b):
            with pytest.raises(E.EpiError):
                x.set_hit_capacity(1 << 40)
        g = s.scan(**kw)
        assert g["nhits"] == want["nhits"] and g["overflow"] and len(g["hits"]) == 0
        st = b.scan(**kw)
        assert st["nhits"] == want["nhits"] and st["overflow"] and b.hits(0)["nhits"] == 0
        for x in (s, b):
            x.set_hit_capacity(1 << 20)
        assert np.array_equal(s.scan(**kw)["hits"], want["hits"])
        b.scan(**kw)
        assert np.array_equal(b.hits(0)["hits"], want["hits"])
