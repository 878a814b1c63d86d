"""128-row tiles of every K-block count, odd ones among them, at each number of
column tiles per workgroup: one-row, full and partial last tiles, unrotated,
rotated in runs of four and not, against the register-staged kernel
(IHE_MFMAW_LDS=0) bit for bit and sampled rows against the oracle (integers mod
2^32: equality)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1024, 512, 333])
@pytest.mark.parametrize("nkb", [2, 3, 4, 5, 6])
def test_every_kblock_count(engine, monkeypatch, nkb, ns):
    for v in ("IHE_CLOUD_KERNEL", "IHE_MFMAW_LDS", "IHE_CLOUD_NTW"):
        monkeypatch.delenv(v, raising=False)
    monkeypatch.setenv("IHE_CLOUD_SHAPE", f"4,{nkb}")
    rng = np.random.default_rng(nkb * 10 + ns)
    width, rows = 32 * nkb, 128 * 3 + 1
    lo = np.repeat([0, 5, 40, 77], [128, 128, 128, 1])      # a tile per window, the last of one row
    num_in = 77 + width + 3
    R = 1024 // ns
    C = (num_in + R - 1) // R
    rp = np.arange(rows + 1, dtype=np.uint32) * width
    ib = (lo[:, None] + np.arange(width)).astype(np.uint32).ravel()
    w = rng.integers(-32768, 32640, ib.size).astype(np.int32)
    ct = rng.integers(-(1 << 31), 1 << 31, (C, 2, 1024), dtype=np.int64).astype(np.int32)
    d_in = engine.to_device(ct)
    got = []
    for lds, ntw in (("0", ""), ("1", "8"), ("2", ""), ("2", "8"), ("2", "16"), ("2", "32")):
        monkeypatch.setenv("IHE_MFMAW_LDS", lds)
        monkeypatch.setenv("IHE_CLOUD_NTW", ntw)
        band = engine.band(ns, C, rp, ib, w)
        info = band.info()
        assert (info["tile_rows"], info["tile_kblocks"], info["num_tiles"]) == (128, nkb, 4)
        d_out = engine.empty((rows, 2, 1024), np.int32)
        engine.cloud(band, d_in, None, d_out, None)
        got.append(d_out.numpy())
        band.free()
        d_out.free()
    for g in got[1:]:
        assert (g == got[0]).all()
    sel = np.array([0, 127, 128, 200, 383, 384])
    pick = (sel[:, None] * width + np.arange(width)).ravel()
    ref, _ = oracle.cloud(ct, np.zeros(C), (np.arange(7) * width).astype(np.uint32), ib[pick],
                          w[pick], ns, R, 1024 // R)
    assert (got[0][sel] == ref).all()
