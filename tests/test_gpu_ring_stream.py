"""Decryptions large enough to take streaming loads of the a-words (98,304
ciphertexts and more at one to three column tiles a wave), the last group
partial, and the largest below, against the VALU kernel: the same floats."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STREAM = 98304


@pytest.fixture(scope="module")
def cts(engine):
    rng = np.random.default_rng(3)
    return engine.to_device(rng.integers(-(1 << 31), 1 << 31, (STREAM + 17, 2, 1024), dtype=np.int32))


@pytest.mark.parametrize("n", [STREAM - 1, STREAM, STREAM + 17])
@pytest.mark.parametrize("ns", [33, 256, 300])
def test_large_decrypt(engine, monkeypatch, cts, n, ns):
    for v in ("IHE_RING_TILES", "IHE_RING_QUEUE", "IHE_DECRYPT_KERNEL"):
        monkeypatch.delenv(v, raising=False)
    k = engine.key(np.random.default_rng(ns).integers(0, 2, 1024).astype(np.int32))
    d_out, d_ref = engine.empty((n, ns), np.float32), engine.empty((n, ns), np.float32)
    d_out.fill_zero()
    engine.decrypt(k, ns, cts, n, d_out)
    monkeypatch.setenv("IHE_DECRYPT_KERNEL", "valu")
    engine.decrypt(k, ns, cts, n, d_ref)
    assert engine.checksum(d_out) == engine.checksum(d_ref)
    k.free()
