"""Bands of one 128-row shape that run different numbers of column tiles join one
launch of a batch; every cohort equals its own launch bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("samples", [(1024, 1024, 700), (200, 512, 256), (100, 333, 77)])
def test_bands_of_different_counts_join(engine, monkeypatch, samples):
    for v in ("IHE_CLOUD_KERNEL", "IHE_MFMAW_LDS", "IHE_BATCH_PERSISTENT"):
        monkeypatch.delenv(v, raising=False)
    monkeypatch.setenv("IHE_CLOUD_SHAPE", "4,3")
    rng = np.random.default_rng(sum(samples))
    width, rows, tags = 96, 128 * 2 + 5, 40
    lo = np.repeat([0, 9, 24], [128, 128, 5])
    rp = np.arange(rows + 1, dtype=np.uint32) * width
    ib = (lo[:, None] + np.arange(width)).astype(np.uint32).ravel()
    cohorts, bands, want = [], [], []
    for ntw, ns in zip(("8", "16", "32"), samples):
        monkeypatch.setenv("IHE_CLOUD_NTW", ntw)
        w = rng.integers(-32768, 32640, ib.size).astype(np.int32)
        bands.append(engine.band(1024, 3 * tags, rp, ib, w))
        assert bands[-1].info()["col_tiles"] == int(ntw)
        C = -(-3 * tags // (1024 // ns))
        d_in = engine.to_device(rng.integers(-(1 << 31), 1 << 31, (C, 2, 1024), dtype=np.int32))
        d_var = engine.to_device(rng.integers(1, 1 << 16, C) * 2.0 ** -60)
        d_out, d_ov = engine.empty((rows, 2, 1024), np.int32), engine.empty((rows,), np.float64)
        cohorts.append((bands[-1], ns, C, d_in, d_var, d_out, d_ov))
        engine.cloud_layout(*cohorts[-1])
        want.append((d_out.numpy(), d_ov.numpy()))
        d_out.fill_zero()
    monkeypatch.delenv("IHE_CLOUD_NTW")
    batch = engine.batch(cohorts)
    assert batch.info()["num_launches"] == 1
    batch.run()
    for c, (o, v) in zip(cohorts, want):
        assert (c[5].numpy() == o).all() and (c[6].numpy() == v).all()
    batch.free()
    for b in bands:
        b.free()
