"""The ring kernel at each number of column tiles per wave (IHE_RING_TILES) and
its own choice: word counts at the edges of column tiles, waves and workgroups,
partial ciphertext groups, and more items than workgroups. Results are integers
(or their exact float conversions), so they are compared for equality."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

TILES = ["1", "2", "3", "4", None]


def set_tiles(monkeypatch, tiles):
    for v in ("IHE_RING_TILES", "IHE_RING_QUEUE", "IHE_ENCRYPT_KERNEL", "IHE_DECRYPT_KERNEL"):
        monkeypatch.delenv(v, raising=False)
    if tiles:
        monkeypatch.setenv("IHE_RING_TILES", tiles)


@pytest.mark.parametrize("tiles", TILES)
@pytest.mark.parametrize("ns", [1, 32, 33, 128, 129, 255, 257, 513, 769, 993, 1023, 1024])
def test_decrypt_tiles(engine, monkeypatch, tiles, ns):
    set_tiles(monkeypatch, tiles)
    rng = np.random.default_rng(ns)
    key = rng.integers(0, 2, 1024).astype(np.int32)
    k = engine.key(key)
    for n in (1, 31, 33, 64):
        cts = rng.integers(-(1 << 31), 1 << 31, (n, 2, 1024)).astype(np.int32)
        cts[0, :, ::3] = -(1 << 31)
        d_in, d_out = engine.to_device(cts), engine.empty((n, ns), np.float32)
        engine.decrypt(k, ns, d_in, n, d_out)
        assert (d_out.numpy() == oracle.decrypt(cts, key, ns)).all(), n
    k.free()


@pytest.mark.parametrize("tiles", TILES)
@pytest.mark.parametrize("n,ns", [(8230, 1024), (8230, 300), (16390, 100), (40, 1024)])
def test_decrypt_items_beyond_the_grid(engine, monkeypatch, tiles, n, ns):
    """Several items per workgroup, the last of them partial, twice in a row (the
    counters are cleared), against the VALU kernel."""
    set_tiles(monkeypatch, tiles)
    rng = np.random.default_rng(n + ns)
    k = engine.key(rng.integers(0, 2, 1024).astype(np.int32))
    d_in = engine.to_device(rng.integers(-(1 << 31), 1 << 31, (n, 2, 1024), dtype=np.int64)
                            .astype(np.int32))
    d_out, d_ref = engine.empty((n, ns), np.float32), engine.empty((n, ns), np.float32)
    engine.decrypt(k, ns, d_in, n, d_out)
    d_out.fill_zero()
    engine.decrypt(k, ns, d_in, n, d_out)
    monkeypatch.setenv("IHE_DECRYPT_KERNEL", "valu")
    engine.decrypt(k, ns, d_in, n, d_ref)
    assert engine.checksum(d_out) == engine.checksum(d_ref)
    k.free()


@pytest.mark.parametrize("tiles", TILES)
@pytest.mark.parametrize("ns,tags", [(1024, 11), (100, 107), (16, 700)])
def test_encrypt_tiles(engine, monkeypatch, tiles, ns, tags):
    set_tiles(monkeypatch, tiles)
    rng = np.random.default_rng(tags)
    geno = rng.integers(-1, 3, (tags, ns)).astype(np.int8)
    key = rng.integers(0, 2, 1024).astype(np.int32)
    R = 1024 // ns
    C = (3 * tags + R - 1) // R
    k = engine.key(key)
    d_geno = engine.to_device(geno)
    d_out, d_var = engine.empty((C, 2, 1024), np.int32), engine.empty((C,), np.float64)
    engine.encrypt(k, ns, d_geno, 5, d_out, d_var)
    ref, rv = oracle.encrypt(geno, key, ns, R, 1024 // R, seed=5)
    assert (d_out.numpy() == ref).all() and (d_var.numpy() == rv).all()
    k.free()
