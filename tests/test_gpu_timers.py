"""The per-kernel timers over IC generation, whose realisation times a fill
inside itself: both are reported with a time, and the report leaves no HIP
error behind for the next call's launch check."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_nested_timers(gev):
    import bbks
    N, h = 32, 0.67
    L = 5.0 * N
    k, d, t = bbks.bbks_table(np.logspace(-5.0, np.log10(300.0), 400), 100.0, 0.31, h)
    sim = gev.SimParams(1, 0, 48.0, 0.04, 100.0, 1.5 * L * L / 2997.92458 ** 2, gev.make_cosmology())
    tpl = gev.load_homogeneous_template(os.path.join(ROOT, "tests", "golden", "sc1_crystal.dat"))
    with gev.Box(N, N ** 3) as b:
        b.timing(True)
        b.generateIC_basic(sim, gev.ICParams(7, 1, 1, N // 4, 100.0, 2.1e-9, 0.965, 0.05, L), tpl, k * L, d, t * L / h, d,
                           t * L / h)
        r = b.timing_report()
        assert r["ic_realize"][0] == 3 and r["ic_realize"][1] > 0.0
        assert all(ms > 0.0 for _, ms in r.values()), r
        b.timing(False)
    with gev.Box(16, 10) as b:  # its first launch check sees no error of the report
        b.synchronize()
