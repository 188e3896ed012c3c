"""The fused cycle on grids on both sides of its size rules (x passes with one
or all tensor components per workgroup, z passes that solve on registers for
powers of two from 64): every carried field and the particles after two cycles
(the second carries B from the first) have the bits of the entry points called
one by one."""
import numpy as np
import pytest

from states import gr_state, sim_params
from test_gpu_parity import cycle_by_calls

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,gr,elliptic,form", [
    (8, True, False, 0), (12, True, False, 0), (24, True, False, 0), (32, False, False, 0), (64, True, False, 0),
    (64, True, True, 0), (64, True, False, 1), (96, True, False, 0), (96, True, False, 1), (128, True, False, 0),
    (128, False, True, 0), (192, True, False, 0), (256, True, False, 0), (256, True, False, 1)])
def test_fused_cycle_has_the_bits_of_the_calls(gev, N, gr, elliptic, form):
    st = gr_state(N, N + 1)
    sp = sim_params(N, 5.0 * N, gr=gr, vector_elliptic=elliptic)
    sim = gev.SimParams(sp["gr_flag"], sp["vector_flag"], sp["Cf"], sp["steplimit"], sp["z_relax"],
                        sp["fourpiG"], gev.make_cosmology())
    a0 = 1.0 / (1.0 + sp["z_in"])
    dt0 = gev.next_dtau(sim, N, a0)
    sg = gev.CycleState(a0, 0.0, dt0, 0.0, 0.0, 0.0, 0.0, 0, 0)
    sc = {"a": a0, "tau": 0.0, "dtau": dt0, "dtau_old": 0.0}
    n = len(st["ids"])
    with gev.Box(N, n, form=form) as fused, gev.Box(N, n, form=form) as calls:
        for b in (fused, calls):
            b.upload_particles(st["pos"], st["q"], st["ids"], st["pmass"])
            for f, key in ((gev.PHI, "phi"), (gev.CHI, "chi"), (gev.BI, "Bi"), (gev.BIFT, "BiFT"),
                           (gev.SCALARFT, "scalarFT")):
                b.upload_field(f, st[key])
        fused.run_cycles(sim, sg, 2)
        for _ in range(2):
            cycle_by_calls(gev, calls, sp, sim, sc)
        assert sg.a == sc["a"] and sg.dtau == sc["dtau"]
        for f in (gev.PHI, gev.CHI, gev.BI, gev.BIFT):
            assert np.array_equal(fused.download_field(f), calls.download_field(f)), f
        for x, y in zip(fused.download_particles(), calls.download_particles()):
            assert np.array_equal(x, y)
