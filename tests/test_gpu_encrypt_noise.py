"""Encryption's a, e and messages (k_encrypt_ae) against the VALU kernel, which
searches the whole noise table for every word, bit for bit: enough words to reach
every length of the search (beyond 3.2 and 3.6 sigma), region sizes that leave
words over and regions that end within a thread's four words, columns that end
within a ciphertext, genotypes outside 0 .. 2, and several ciphertexts per
workgroup. Integers mod 2^32: equality."""
import ctypes

import numpy as np
import pytest

from idash2019_2_amd import _abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,tags", [
    (1024, 2500), (1021, 3), (341, 1201), (300, 700), (5, 4001), (2, 1500), (1, 5000), (3, 1234)])
def test_matches_full_search(engine, monkeypatch, ns, tags):
    R = 1024 // ns
    rs = 1024 // R
    for v in ("IHE_RING_TILES", "IHE_RING_QUEUE", "IHE_ENCRYPT_KERNEL"):
        monkeypatch.delenv(v, raising=False)
    rng = np.random.default_rng(tags + ns)
    geno = rng.integers(0, 3, (tags, ns)).astype(np.int8)
    odd = rng.random((tags, ns)) < 0.01
    geno[odd] = rng.integers(-128, 128, int(odd.sum()))
    C = (3 * tags + R - 1) // R
    k = engine.key(rng.integers(0, 2, 1024).astype(np.int32))
    d_geno = engine.to_device(geno)
    lay = _abi.Layout(ns, R, rs)
    for g in (d_geno.ptr, None):
        got = []
        for kernel in ("", "valu"):
            monkeypatch.setenv("IHE_ENCRYPT_KERNEL", kernel)
            d_out, d_var = engine.empty((C, 2, 1024), np.int32), engine.empty((C,), np.float64)
            _abi.check(_abi.lib().ihe_encrypt(engine.ctx, k.handle, ctypes.byref(lay), tags, g,
                                              1234567 + ns, d_out.ptr, d_var.ptr))
            got.append((d_out.numpy(), d_var.numpy()))
            d_out.free()
            d_var.free()
        assert (got[0][0] == got[1][0]).all() and (got[0][1] == got[1][1]).all()
    k.free()
