"""The filing on grids on both sides of its size rules (partials of the scan
added up by every block or scanned first; segments of the ID sort spread over
the chip or 32 to a workgroup): per-cell counts, and the cell-sorted order
with ascending IDs that a drift stores, against numpy.  Clustered particles,
so that every tier of the sort has cells: one, up to 4, up to a segment's LDS
and above it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,n", [(12, 5000), (48, 60000), (128, 300000), (192, 300000), (256, 300000)])
def test_counts_and_order(gev, N, n):
    rng = np.random.default_rng(N)
    pos = rng.random((n, 3))
    m = n // 3
    pos[:m] = (rng.random((40, 3))[rng.integers(0, 40, m)] + 0.6 / N * rng.standard_normal((m, 3))) % 1.0
    pos[m:m + 1500] = 0.5 + 0.8 / N * rng.random((1500, 3))  # a cell of at least 1500
    pos[pos >= 1.0] = 0.0
    ids = rng.permutation(n).astype(np.int64)
    ci = np.floor(pos / (1.0 / N)).astype(np.int64)
    cell = ci[:, 0] + N * (ci[:, 1] + N * ci[:, 2])
    with gev.Box(N, n) as b:
        b.upload_particles(pos, np.zeros((n, 3)), ids, 1.0)
        for _ in range(2):  # a second filing from the stored order
            counts, cells = b.download_filing()
            assert np.array_equal(counts, np.bincount(cell, minlength=N ** 3))
            # no momentum: the particles stay and are stored in the order of the filing
            b.moveParticles(gev.POS_NEWTON, 0.1, 0, [0.5, 0.25 * N])
            p, _, i = b.download_particles()
            o = np.lexsort((ids, cell))
            assert np.array_equal(i, ids[o])
            assert np.array_equal(p, pos[o])


def _wide_ids(rng, n, kind):
    ids = rng.permutation(n).astype(np.int64)
    if kind == "edge":  # the largest ID of the 32-bit comparison and the first beyond it
        ids += 2 ** 32 - 2 - n // 2
    elif kind == "mixed":  # beyond 32 bits with equal low words, negative, repeated
        w = rng.random(n) < 0.3
        ids[w] += rng.integers(-3, 4, w.sum()) << 32
        ids[rng.integers(0, n, 50)] = ids[rng.integers(0, n, 50)]
    else:  # every ID several times
        ids //= 5
    return ids


@pytest.mark.parametrize("kind", ["edge", "mixed", "repeated"])
def test_order_by_wide_and_repeated_ids(gev, kind):
    N, n = 48, 60000
    rng = np.random.default_rng(len(kind))
    pos = rng.random((n, 3))
    pos[:20000] = (rng.random((40, 3))[rng.integers(0, 40, 20000)] + 0.3 / N * rng.standard_normal((20000, 3))) % 1.0
    pos[20000:21500] = 0.5 + 0.8 / N * rng.random((1500, 3))
    pos[pos >= 1.0] = 0.0
    ids = _wide_ids(rng, n, kind)
    ci = np.floor(pos / (1.0 / N)).astype(np.int64)
    cell = ci[:, 0] + N * (ci[:, 1] + N * ci[:, 2])
    o = np.lexsort((ids, cell))
    with gev.Box(N, n) as b:
        b.upload_particles(pos, np.zeros((n, 3)), ids, 1.0)
        b.moveParticles(gev.POS_NEWTON, 0.1, 0, [0.5, 0.25 * N])
        p, _, i = b.download_particles()
    assert np.array_equal(i, ids[o])
    assert np.array_equal(np.sort(p, axis=0), np.sort(pos, axis=0))
    # particles of one cell and ID may come in any order, others not
    new = np.append(True, (np.diff(ids[o]) != 0) | (np.diff(cell[o]) != 0))
    u = new & np.append(new[1:], True)
    assert np.array_equal(p[u], pos[o][u])
