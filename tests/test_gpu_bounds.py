"""The harmonic sum by bounds (k_harmbound) against the sums themselves:
every hit recomputed in numpy from the search's raw plane and norms, term by
term in FP32 in the order of the fractions, so set and powers must be equal.
The shapes are those at which it can go wrong: 1 to 5 stages, both index
rules, one, two and four blocks of z rows, jerk rows, ragged lengths, a first
half-bin off every chunk edge, a last one inside a run, strong signals, bins
without power, infinities and NaN.  The handle says which kernel it runs."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
A = pytest.importorskip("presto_amd.accel")


def _by_bounds(s):
    """Whether k_harmbound runs, as the handle itself says."""
    A.lib.accel_search_uses_bounds.argtypes = [C.c_void_p]
    return A.lib.accel_search_uses_bounds(s.h) == 1


def _nearest(x):
    return np.where(x < 0, np.ceil(x - 0.5), np.floor(x + 0.5)).astype(int)


def _expected(s):
    g = s.geom
    numw = max(g.numw, 1)
    ncell = g.nblocks * g.corr_uselen
    rh0 = 2 * int(np.floor(np.rint(2 * g.rlo) / 2))
    plane = np.stack([np.stack([s.plane_row(w, z, 0, rh0 + ncell) for z in range(g.numz)])
                      for w in range(numw)])
    norm = s.norms()
    nsq = (norm * norm).astype(np.float32)
    rh = rh0 + np.arange(ncell)
    block = np.arange(ncell) // g.corr_uselen
    if g.inmem:
        npre = len(norm) - g.nblocks
        hb = np.arange(rh0 + ncell)
        owner = np.where(hb >= rh0, npre + (hb - rh0) // g.corr_uselen, (hb - 16) // g.corr_uselen)
        nsq_hb = np.where((hb < 16) & (hb < rh0), np.float32(0), nsq[owner.clip(0)])
    nfr = 1 << (g.numharmstages - 1)
    zs = g.zlo + 2.0 * np.arange(g.numz)
    ws = g.wlo + 20.0 * np.arange(numw)
    hits = []
    acc, f = None, 0
    for st in range(g.numharmstages):
        H = 1 << st
        for k in range(1, H + (st == 0), 2):
            q = rh * k
            rs = (q + H // 2) // H if g.inmem else np.rint(q / H).astype(np.int64)
            zi = ((2 * _nearest(0.5 * zs * k / H) + g.zhi) / 2).astype(int)
            wi = ((20 * _nearest(0.05 * ws * k / H) + g.whi) / 20).astype(int) if g.numw else [0]
            n = nsq_hb[rs] if g.inmem else nsq.reshape(g.nblocks, nfr)[block, f]
            with np.errstate(all="ignore"):
                term = plane[np.ix_(wi, zi)][:, :, rs] * n
                acc = term if acc is None else acc + term
            f += 1
        with np.errstate(all="ignore"):
            for w, z, c in np.argwhere(acc > np.float32(g.powcut[st])):
                hits.append((int(c) // g.corr_uselen, st, int(w), int(z), int(c) % g.corr_uselen,
                             acc[w, z, c]))
    return sorted(hits, key=lambda h: h[:5])


def _spectrum(nbins, seed, signals=(), odd=None):
    rng = np.random.Generator(np.random.PCG64(seed))
    X = (rng.standard_normal(nbins) + 1j * rng.standard_normal(nbins)) / np.sqrt(2.0)
    for r, amp in signals:
        X[r] += amp
    X = X.astype(np.complex64)
    X[0] = 1 + 1j
    if odd == "zeros":
        X[nbins // 2:nbins // 2 + 6000] = 0
    if odd == "inf":
        X[nbins // 2] = np.inf
        X[nbins // 3] = complex(np.nan, 1.0)
    return X


@pytest.mark.parametrize("nbins,zmax,wmax,numharm,inmem,rlo,odd", [
    (150000, 30, None, 1, False, 100, None),
    (150000, 30, None, 2, True, 101, None),
    (100001, 63, None, 4, False, 333, None),          # 64 rows, one block
    (100001, 64, None, 4, True, 333, None),           # 65 rows, two
    (1 << 17, 50, None, 8, True, 21, None),
    (1 << 17, 50, None, 8, False, 22, "zeros"),
    (1 << 17, 50, None, 8, True, 23, "inf"),
    (1 << 17, 50, None, 8, False, 23, "inf"),
    (1 << 18, 100, None, 16, False, 77, None),
    (1 << 18, 100, None, 16, True, 1, None),
    (60000, 30, 40, 8, False, 50, None),              # 31 x 5 rows
    (45001, 200, None, 8, True, 50, None),            # 201 rows, four blocks of 51 or 48
    (45001, 200, None, 16, False, 50, None),
])
def test_hits_equal_the_sums(nbins, zmax, wmax, numharm, inmem, rlo, odd):
    sig = [(nbins // 7, 9.0), (2 * (nbins // 7), 8.0), (3 * (nbins // 7), 7.0),
           (nbins // 5 + 3, 200.0), (rlo + 5, 12.0)]
    p = A.make_params(nbins, 2 * nbins, 1e-3, zmax=zmax, numharm=numharm, sigma=2.5, wmax=wmax,
                      rlo=rlo, rhi=nbins - 1, inmem=inmem, force_standard=not inmem,
                      dat_input=False)
    with A.Search(p) as s:
        assert _by_bounds(s) and bool(s.geom.inmem) == inmem
        s.set_spectrum(_spectrum(nbins, 11 + numharm, sig, odd))
        s.run()
        got = [(int(h["block"]), int(h["stage"]), int(h["wi"]), int(h["zi"]), int(h["ii"]),
                h["pow"]) for h in s.hits()]
        want = _expected(s)
    assert len(want) > 20
    assert [h[:5] for h in got] == [h[:5] for h in want]
    np.testing.assert_array_equal(np.array([h[5] for h in got]), np.array([h[5] for h in want]))


@pytest.fixture
def used_memory():
    """Device memory whose last user left a large negative number in every
    word (0xfefe...): an arena, as the request loop's handles share one."""
    lib, n, p = A.lib, 1 << 30, C.c_void_p()
    lib.agpu_malloc.argtypes = [C.c_void_p, C.c_size_t]
    lib.agpu_memset.argtypes = [C.c_void_p, C.c_int, C.c_size_t, C.c_void_p]
    lib.agpu_free.argtypes = lib.agpu_stream_sync.argtypes = [C.c_void_p]
    lib.agpu_arena_init.argtypes = [C.c_size_t]
    lib.accel_template_cache_clear()
    assert lib.agpu_init(0) == 0 and lib.agpu_arena_init(n) == 0
    assert lib.agpu_malloc(C.byref(p), n) == 0 and lib.agpu_memset(p, 0xfe, n, None) == 0
    assert lib.agpu_stream_sync(None) == 0 and lib.agpu_free(p) == 0
    yield
    lib.accel_template_cache_clear()
    assert lib.agpu_arena_release() == 0


@pytest.mark.parametrize("numharm,inmem", [(1, False), (8, True), (16, False)])
def test_the_last_half_bins_in_used_memory(used_memory, numharm, inmem):
    """A signal in the last, partial run of 64 half-bins, whose other bounds
    no correlation writes."""
    nbins, rlo = (150000, 110) if numharm < 16 else (1 << 18, 77)
    p = A.make_params(nbins, 2 * nbins, 1e-3, zmax=30 if numharm < 16 else 100, numharm=numharm,
                      sigma=2.5, rlo=rlo, rhi=nbins - 1, inmem=inmem, force_standard=not inmem,
                      dat_input=False)
    g = A.geometry(p)
    end = 2 * int(np.floor(np.rint(2 * g.rlo) / 2)) + g.nblocks * g.corr_uselen
    run = end // 64 * 64
    assert 16 <= end - run <= 48
    with A.Search(p) as s:
        assert _by_bounds(s)
        s.set_spectrum(_spectrum(nbins, 5, [(run // 2 + 2, 40.0)]))
        s.run()
        got = [(int(h["block"]), int(h["stage"]), int(h["wi"]), int(h["zi"]), int(h["ii"]),
                h["pow"]) for h in s.hits()]
        want = _expected(s)
    assert sum(h[0] * g.corr_uselen + h[4] + end - g.nblocks * g.corr_uselen >= run
               for h in want) > 5
    assert got == want


@pytest.mark.parametrize("bits", [0x7fffffff, 0xffffffff, 0x7fc00000])
def test_nan_beside_a_signal(bits):
    """A NaN, whatever its payload and sign, fills one segment of the
    correlation; the signal lies in the next one, in the same run of 64
    half-bins."""
    nbins = 150000
    p = A.make_params(nbins, 2 * nbins, 1e-3, zmax=40, numharm=1, sigma=2.5, rlo=100,
                      rhi=nbins - 1, force_standard=True, dat_input=False)
    with A.Search(p) as s:
        assert _by_bounds(s)
        uselen = s.corr_shape()["uselen"]
        hw = (4096 - uselen) // 4
        end = next(e for e in range(20 * uselen, 60 * uselen, uselen) if 16 <= e % 64 <= 48)
        X = _spectrum(nbins, 6, [(end // 2 + 2, 40.0)])
        bad = (end - uselen) // 2 + hw + 10   # in reach of no other segment
        X.view(np.uint32)[2 * bad:2 * bad + 2] = bits
        s.set_spectrum(X)
        s.run()
        got = [(int(h["block"]), int(h["stage"]), int(h["wi"]), int(h["zi"]), int(h["ii"]),
                h["pow"]) for h in s.hits()]
        want = _expected(s)
        for z in range(s.geom.numz):
            assert np.isnan(s.plane_row(0, z, end - 4, 4)).all()
            assert np.isfinite(s.plane_row(0, z, end, 4)).all()
    near = [h for h in want
            if end <= 200 + h[0] * s.geom.corr_uselen + h[4] < (end // 64 + 1) * 64]
    assert len(near) > 5 and got == want


@pytest.mark.parametrize("kw", [
    dict(numharm=32), dict(zmax=14, nbins=300000), dict(nbins=60000), dict(sigma=1.0, numharm=16),
    dict(rlo=100.5), dict(rlo=100.25)])
def test_searches_that_sum_every_cell(kw):
    """32 harmonics, 15 rows (one less than the rule asks), few cells, a low
    threshold and starts off whole bins do not take the bounds; the in-memory
    rule takes no half-bin start's lookups, so that one does."""
    nbins = kw.pop("nbins", 150000)
    kw = dict(dict(zmax=30, numharm=8, sigma=2.5, rlo=100), **kw)
    p = A.make_params(nbins, 2 * nbins, 1e-3, rhi=nbins - 1, force_standard=True,
                      dat_input=False, **kw)
    with A.Search(p) as s:
        assert s.geom.numz == kw["zmax"] + 1 and not _by_bounds(s)
    if kw["rlo"] == 100.5:
        p.force_standard, p.inmem = 0, 1
        with A.Search(p) as s:
            assert s.geom.inmem and _by_bounds(s)
