"""The batch's tile autotuner times the y pass by the launches of a cycle, on
the batch's own fields, and leaves every field of every box as it was; its
times are per component, and a second call repeats the picks."""
import numpy as np
import pytest

from states import gr_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nbox,form", [(96, 5, 0), (96, 5, 1)])
def test_autotune(gev, N, nbox, form):
    rng = np.random.default_rng(N + form)
    s = gr_state(N, 5)
    n = len(s["ids"])
    sijft = (rng.standard_normal((6, N, N, N // 2 + 1)) + 1j * rng.standard_normal((6, N, N, N // 2 + 1)))
    with gev.Batch(N, n, nbox, gr=1, form=form) as B:
        views = [B.box(i) for i in (0, 2, nbox - 1)]
        fields = (gev.PHI, gev.CHI, gev.BI, gev.BIFT, gev.SCALARFT, gev.SIJFT, gev.SIJ, gev.SOURCE)
        for j, v in enumerate(views):
            v.upload_field(gev.SIJFT, sijft * (1 + j))
            v.upload_field(gev.BIFT, s["BiFT"] * (1 + j))
            v.upload_field(gev.PHI, s["phi"] * (1 + j))
        before = [[v.download_field(f) for f in fields] for v in views]
        t = B.autotune()
        for v, old in zip(views, before):
            for f, x in zip(fields, old):
                assert np.array_equal(v.download_field(f), x), f
        assert t["y_row_bytes"] in (64, 128, 256) and t["z_row_bytes"] in (64, 128, 256)
        print("y %s z %s" % tuple(t["pass_ms"]), flush=True)
        assert all(ms > 0.0 for axis in t["pass_ms"] for ms in axis)
        assert B.autotune() == t
