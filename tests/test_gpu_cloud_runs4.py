"""The one-K-block cloud kernel with 16-byte loads and stores, on both sides of
every line of its dispatch (bytes written; unrotated and rotated layouts; words
in runs of four or not) against the dword kernel (IHE_CLOUD_NTW=8), bit for bit,
and sampled rows against the oracle. Integers mod 2^32: equality."""
import numpy as np
import pytest

import oracle
from idash2019_2_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,targets", [
    (1024, 40), (1024, 1901), (1024, 2100), (1024, 6500), (1024, 7000), (1000, 7001),
    (512, 5100), (512, 5600), (200, 5601), (16, 5600), (333, 2000), (100, 5600)])
def test_runs_of_four_match_dword_kernel(engine, monkeypatch, ns, targets):
    for v in ("IHE_CLOUD_SHAPE", "IHE_CLOUD_KERNEL", "IHE_CLOUD_NTW"):
        monkeypatch.delenv(v, raising=False)
    monkeypatch.setenv("IHE_CLOUD_SHAPE", "2,1")
    tags = 40 + targets // 5
    rng = np.random.default_rng(targets + ns)
    lo = np.sort(rng.integers(0, tags - 5 + 1, targets))
    cols = np.repeat(3 * lo, 3)[:, None] + np.arange(15)
    ib = np.concatenate([cols, np.full((3 * targets, 1), synth.CONSTANT_BIDX)], axis=1)
    w = rng.integers(-32768, 32640, ib.shape).astype(np.int32)
    rp = np.arange(3 * targets + 1, dtype=np.uint32) * 16
    ib, w = ib.astype(np.uint32).ravel(), w.ravel()
    R = 1024 // ns
    C = (3 * tags + R - 1) // R
    ct = rng.integers(-(1 << 31), 1 << 31, (C, 2, 1024), dtype=np.int64).astype(np.int32)
    var = rng.random(C) * 2.0 ** -40
    d_in, d_var = engine.to_device(ct), engine.to_device(var)
    sums = []
    for ntw in (None, "8"):
        if ntw:
            monkeypatch.setenv("IHE_CLOUD_NTW", ntw)
        band = engine.band(ns, C, rp, ib, w)
        assert (band.info()["tile_rows"], band.info()["tile_kblocks"]) == (64, 1)
        d_out = engine.empty((3 * targets, 2, 1024), np.int32)
        d_ov = engine.empty((3 * targets,), np.float64)
        d_out.fill_zero()
        engine.cloud(band, d_in, d_var, d_out, d_ov)
        sums.append((engine.checksum(d_out), engine.checksum(d_ov)))
        if not ntw:
            rows = np.unique(np.r_[0, 3 * targets - 1, rng.integers(0, 3 * targets, 6)])
            got = d_out.take(rows)
        band.free()
        d_out.free()
    assert sums[0] == sums[1]
    rp_s = (np.arange(rows.size + 1) * 16).astype(np.uint32)
    sel = (rows[:, None] * 16 + np.arange(16)).ravel()
    ref, _ = oracle.cloud(ct, var, rp_s, ib[sel], w[sel], ns, R, 1024 // R)
    assert (got == ref).all()
