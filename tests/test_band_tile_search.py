"""The band compiler's shape search against a restatement of its rule in Python:
greedy tiles of at most 32 rb rows and 32 nkb distinct columns, the shape of least
estimated time, column tiles by the tile count. Dense columns, and columns so
sparse that they are counted by rank; rows without columns among them."""
import numpy as np
import pytest

from idash2019_2_amd import engine


def greedy(rows, rb, nkb):
    tiles, o = 0, 0
    while o < len(rows):
        cols, o0 = set(), o
        while o < len(rows) and o - o0 < 32 * rb and len(cols | rows[o]) <= 32 * nkb:
            cols |= rows[o]
            o += 1
        if o == o0:
            return 0
        tiles += 1
    return tiles


def expected(rows):
    kmin = max(1, -(-max(len(r) for r in rows) // 32))
    shapes = [(2, 1), (1, 1)] if kmin == 1 else []
    shapes += [(1, k) for k in range(max(2, kmin), min(kmin + 2, 8) + 1)]
    wide, k = [], max(2, kmin)
    while k <= min(kmin + 3, 8):
        wide.append((4, k + (k == 7)))
        k += 1 if k < 6 else 2
    best = None
    for rb, k in shapes + wide:
        t = greedy(rows, rb, k)
        cost = t * (3.2 * k + 4.5) if rb == 4 else t * (k + 1.5 * rb)
        if t and (best is None or cost < best[0]):
            best = (cost, rb, k, t)
    _, rb, k, t = best
    ntw = 4 if rb != 4 else 32 if k > 6 else 8 if t < (100 if k <= 2 else 200) else \
        32 if k > 2 and t >= 900 else 16
    return 32 * rb, k, t, ntw


@pytest.mark.parametrize("stride", [1, 997])
@pytest.mark.parametrize("n,targets", [(5, 60), (11, 700), (22, 300), (33, 2500), (53, 200), (72, 90)])
def test_shape_search(monkeypatch, n, targets, stride):
    for v in ("IHE_CLOUD_SHAPE", "IHE_CLOUD_KERNEL", "IHE_CLOUD_NTW"):
        monkeypatch.delenv(v, raising=False)
    rng = np.random.default_rng(n + stride)
    start = np.sort(rng.integers(0, targets // 4 + 1, targets))
    rows = []
    for lo in start:
        drop = rng.random(3 * n) < 0.1
        rows += [set(((3 * lo + np.arange(3 * n)[~drop]) * stride).tolist())] * 3
    rows[4] = set()
    rp = np.cumsum([0] + [len(r) for r in rows]).astype(np.uint32)
    ib = np.concatenate([np.sort(np.array(list(r), np.int64)) for r in rows]).astype(np.uint32)
    info = engine.band_plan(1024, int(ib.max()) + 1, rp, ib, np.ones(ib.size, np.int32))
    assert (info["tile_rows"], info["tile_kblocks"], info["num_tiles"], info["col_tiles"]) == expected(rows)
