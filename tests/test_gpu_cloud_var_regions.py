"""Output variances over many ciphertexts at every kind of region count (1, powers
of two, others): rows of 0 to 33 entries around the groups that a wave takes at a
time, columns at the first regions of high-numbered ciphertexts and beside them,
weights in 16 bits and wider (packed and plain entries). All rows with finite
variances first, then the rows that a ciphertext without a finite variance does
not enter. Variances are small integers times one power of two, so that the sums
are exact in double and compared for equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C, FIRST = 4001, 3941                # ciphertexts; the rows use the last 60
COUNTS = [0, 1, 7, 8, 9, 15, 16, 17, 24, 33]


@pytest.mark.parametrize("largest", [2000, 40000])
@pytest.mark.parametrize("ns", [1024, 512, 341, 100, 16, 1])
def test_variances_of_many_ciphertexts(engine, ns, largest):
    rng = np.random.default_rng(ns + largest)
    R = 1024 // ns
    heads = np.arange(FIRST, C) * R
    pool = np.unique(np.concatenate([heads, heads[1:] - 1, heads[:-1] + R // 2]))
    counts = np.resize(COUNTS, 131)
    rows = [rng.permutation(pool)[:n] if i % 2 else rng.permutation(heads)[:n]
            for i, n in enumerate(counts)]
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    ib = np.concatenate(rows).astype(np.uint32)
    w = rng.integers(-largest, largest + 1, ib.size).astype(np.int32)
    w[0] = largest                   # one weight beyond 16 bits makes the entries plain
    var = rng.integers(1, 1000, C) * 2.0 ** -50
    band = engine.band(ns, C, rp, ib, w)
    d_in, d_out = engine.empty((C, 2, 1024), np.int32), engine.empty((131, 2, 1024), np.int32)
    d_in.fill_zero()
    d_ov = engine.empty((131,), np.float64)
    for hole, value in ((None, 0.0), (3977, np.inf), (3950, np.nan)):
        v = var.copy()
        if hole is not None:
            v[hole] = value
        engine.cloud(band, d_in, engine.to_device(v), d_out, d_ov)
        got, seen = d_ov.numpy(), set()
        for o, cols in enumerate(rows):
            kept = cols % R == 0
            if hole is not None and (cols[kept] // R == hole).any():
                continue
            ww = w[rp[o]:rp[o + 1]][kept].astype(np.float64)
            assert got[o] == (ww * ww * v[cols[kept] // R]).sum(), (o, hole)
            if kept.any():
                seen.add(len(cols))
        assert seen >= {7, 8, 9, 15, 16, 17}, (hole, seen)
    band.free()
