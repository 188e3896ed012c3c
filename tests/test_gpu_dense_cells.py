"""Cells of more particles than the filing ranks in LDS (2048), sorted in
place: the stored order is by cell and ID, with ties of equal IDs by storage
index, in a single box and in boxes of a batch that hold different numbers of
such cells; and they cost no more than a small multiple of the cells below
that limit (one thread per cell once took 14 ms each)."""
import numpy as np
import pytest

from states import gr_state, sim_params

pytestmark = pytest.mark.gpu


def dense(N, sizes, seed, spare=500):
    """Particles in len(sizes) cells of the given counts and spare others."""
    rng = np.random.default_rng(seed)
    cells = rng.choice(N ** 3, len(sizes), replace=False)
    c = np.stack([cells % N, cells // N % N, cells // N // N], axis=1)
    n = int(sum(sizes))
    pos = np.concatenate([(np.repeat(c, sizes, axis=0) + 0.01 + 0.98 * rng.random((n, 3))) / N,
                          rng.random((spare, 3))])
    o = rng.permutation(len(pos))
    pos = np.ascontiguousarray(pos[o])
    pos[pos >= 1.0] = 0.0
    ci = np.floor(pos / (1.0 / N)).astype(np.int64)
    return pos, ci[:, 0] + N * (ci[:, 1] + N * ci[:, 2]), rng


@pytest.mark.parametrize("kind", ["plain", "wide", "repeated"])
@pytest.mark.parametrize("N,sizes", [(8, [2047, 2048, 2049, 2050]), (32, [2049, 4096, 4097, 5001, 700, 9])])
def test_order(gev, N, sizes, kind):
    pos, cell, rng = dense(N, sizes, N)
    n = len(pos)
    ids = rng.permutation(n).astype(np.int64)
    if kind == "wide":
        ids += np.int64(2) ** 33 * rng.integers(-1, 2, n)
    elif kind == "repeated":
        ids //= 7
    o = np.lexsort((np.arange(n), ids, cell))
    with gev.Box(N, n) as b:
        b.upload_particles(pos, np.zeros((n, 3)), ids, 1.0)
        b.moveParticles(gev.POS_NEWTON, 0.1, 0, [0.5, 0.25 * N])
        p, _, i = b.download_particles()
    assert np.array_equal(i, ids[o])
    # ties by storage index hold above the LDS limit; below it equal IDs of one cell may come in any order
    big = np.bincount(cell, minlength=N ** 3)[cell[o]] > 2048
    u = big | (kind != "repeated")
    assert big.any() and np.array_equal(p[u], pos[o][u])


def test_time(gev):
    pos, cell, rng = dense(32, [2500] * 24, 5)
    n = len(pos)
    with gev.Box(32, n) as b:
        b.upload_particles(pos, np.zeros((n, 3)), rng.permutation(n).astype(np.int64), 1.0)
        b.timing(True)
        b.moveParticles(gev.POS_NEWTON, 0.1, 0, [0.5, 8.0])
        ms = b.timing_report()["filing_sort_dense_cells"][1]
    print("24 cells of 2500 particles: %.2f ms" % ms, flush=True)
    assert ms < 50.0


@pytest.mark.parametrize("form", [0, 1])
def test_batch(gev, form):
    """Boxes with none, a few and many dense cells, one of them switched off:
    fields and particles of each equal those of the box run alone."""
    N, nbox = 16, 4
    sizes = [[], [2100] * 3, [3000] * 40, [2500] * 12]
    n = 121000
    sp = sim_params(N, 5.0 * N)
    sim = gev.SimParams(sp["gr_flag"], sp["vector_flag"], sp["Cf"], sp["steplimit"], sp["z_relax"], sp["fourpiG"],
                        gev.make_cosmology())
    a0 = 1.0 / 101.0
    fields = gr_state(N, 3)

    def fill(b, i):
        pos, _, rng = dense(N, sizes[i], 10 + i, spare=n - int(sum(sizes[i])))
        b.upload_particles(pos, 1e-6 * rng.standard_normal((n, 3)), rng.permutation(n).astype(np.int64), 0.31 / n)
        for f, k in ((gev.PHI, "phi"), (gev.CHI, "chi"), (gev.BI, "Bi"), (gev.BIFT, "BiFT"),
                     (gev.SCALARFT, "scalarFT")):
            b.upload_field(f, fields[k])

    def state():
        return gev.CycleState(a0, 0.0, gev.next_dtau(sim, N, a0), 0.0, 0.0, 0.0, 0.0, 0, 0)

    with gev.Batch(N, n, nbox, gr=1, form=form) as B:
        for i in range(nbox):
            fill(B.box(i), i)
            B.start_box(i, sim, state(), 5.0 * N)
        B.run_cycles(1)
        B.stop_box(1)
        B.run_cycles(2)
        for i in range(nbox):
            with gev.Box(N, n, form=form) as b:
                fill(b, i)
                b.run_cycles(sim, state(), 1 if i == 1 else 3)
                for f in (gev.PHI, gev.CHI, gev.BI):
                    assert np.array_equal(B.box(i).download_field(f), b.download_field(f)), (i, f)
                for x, y in zip(B.box(i).download_particles(), b.download_particles()):
                    assert np.array_equal(x, y), i
