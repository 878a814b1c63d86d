"""Output variances of the cloud step: rows whose entry counts lie around the
group of entries that a wave takes at a time, every kind of region count (1,
powers of two, others), and non-finite input variances in columns that a row
does not use. Variances are small integers times one power of two, so the
products and sums are exact in double and compared for equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1024, 512, 341, 100, 16, 1])
@pytest.mark.parametrize("tags", [1, 2, 3, 5, 6, 16])
def test_variances_of_short_and_long_rows(engine, ns, tags):
    rng = np.random.default_rng(ns + tags)
    R = 1024 // ns
    num_in = 3 * tags
    C = (num_in + R - 1) // R
    outputs = 131
    rows = []
    for o in range(outputs):  # 0 .. all columns, in any order, and a constant
        n = int(rng.integers(0, num_in + 1))
        rows.append(rng.permutation(num_in)[:n])
    rp = np.concatenate([[0], np.cumsum([r.size + 1 for r in rows])]).astype(np.uint32)
    ib = np.concatenate([np.append(r, 0xFFFFFFFF) for r in rows]).astype(np.uint32)
    w = rng.integers(-2000, 2001, ib.size).astype(np.int32)
    var = rng.integers(0, 1000, C) * 2.0 ** -50
    hole = int(rng.integers(0, C))                  # a ciphertext with no finite variance,
    rows_ok = [o for o in range(outputs) if not (rows[o] // R == hole).any()]
    var[hole] = np.inf
    band = engine.band(ns, C, rp, ib, w)
    d_in = engine.to_device(np.zeros((C, 2, 1024), np.int32))
    d_out = engine.empty((outputs, 2, 1024), np.int32)
    d_ov = engine.empty((outputs,), np.float64)
    engine.cloud(band, d_in, engine.to_device(var), d_out, d_ov)
    got = d_ov.numpy()
    for o in rows_ok:                               # which the rows that do not use it never see
        want = sum(float(w[rp[o] + i]) ** 2 * var[c // R]
                   for i, c in enumerate(rows[o]) if c % R == 0)
        assert got[o] == want, (o, got[o], want)
    band.free()
