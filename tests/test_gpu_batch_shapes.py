"""Batches at the sizes where the launches over boxes take another path than a
small batch's: the z pass that solves on registers with boxes (FP64, 64^3 and
128^3), the tensor x pass with six components per workgroup and boxes (32^3
from 16 boxes on, 96^3; over twice the rows with 40 boxes of 32^3, 57 of 24^3, 8
of 48^3, 5 of 64^3), one component per workgroup just below that line,
column passes over components and boxes, radix-3 grids.  Boxes of different
states, one stopped after the first cycle, graph replay and plain launches:
every carried field and the particles of each equal those of the box run
alone, bit for bit."""
import numpy as np
import pytest

from states import gr_state, sim_params

pytestmark = pytest.mark.gpu

FIELDS = ("phi", "chi", "Bi", "BiFT", "scalarFT")


def setup(gev, N, i, gr):
    sp = sim_params(N, (4.0 + 0.1 * i) * N, gr=bool(gr))
    sim = gev.SimParams(sp["gr_flag"], sp["vector_flag"], sp["Cf"], sp["steplimit"], sp["z_relax"], sp["fourpiG"],
                        gev.make_cosmology(0.25 + 0.002 * i))
    a0 = 1.0 / (101.0 - 0.5 * i)
    return sim, gev.CycleState(a0, 0.0, gev.next_dtau(sim, N, a0), 0.0, 0.0, 0.0, 0.0, 0, 0), sp


def fill(gev, box, s, i):
    # a state of its own for every box: the shared one, shifted and scaled
    pos = np.mod(s["pos"] + 0.137 * i, 1.0)
    pos[pos >= 1.0] = 0.0
    box.upload_particles(pos, s["q"] * (1.0 + 0.01 * i), s["ids"][::-1].copy() if i % 2 else s["ids"], s["pmass"])
    for f, k in zip((gev.PHI, gev.CHI, gev.BI, gev.BIFT, gev.SCALARFT), FIELDS):
        box.upload_field(f, s[k] * (1.0 - 0.02 * i))


@pytest.mark.parametrize("N,nbox,form,gr", [
    (32, 15, 0, 1), (32, 17, 0, 1), (32, 17, 1, 1), (32, 66, 1, 0), (32, 40, 0, 1), (24, 57, 0, 1), (48, 3, 0, 1), (48, 8, 0, 1), (64, 5, 0, 1), (64, 3, 0, 1), (64, 2, 1, 1),
    (96, 2, 0, 1), (96, 2, 1, 1), (128, 2, 0, 1), (192, 2, 0, 1)])
def test_boxes_equal_alone(gev, N, nbox, form, gr):
    s = gr_state(N, N + nbox)
    n, off = len(s["ids"]), nbox // 2
    with gev.Batch(N, n, nbox, gr=gr, form=form) as B:
        for i in range(nbox):
            fill(gev, B.box(i), s, i)
            sim, st, sp = setup(gev, N, i, gr)
            B.start_box(i, sim, st, sp["N"] * 5.0)
        B.run_cycles(1, graph=False)
        B.stop_box(off)
        B.run_cycles(2, graph=True)
        for i in sorted({0, 1, off, nbox - 1}):
            with gev.Box(N, n, form=form) as b:
                fill(gev, b, s, i)
                sim, st, _ = setup(gev, N, i, gr)
                b.run_cycles(sim, st, 1 if i == off else 3)
                for f in (gev.PHI, gev.CHI, gev.BI, gev.BIFT):
                    assert np.array_equal(B.box(i).download_field(f), b.download_field(f)), (i, f)
                for x, y in zip(B.box(i).download_particles(), b.download_particles()):
                    assert np.array_equal(x, y), i
