"""What a user of the library has it do, as measurable cases.

Every case goes through the Python binding (gevolution-1.2_amd/gevpm.py) as a
program of a user does: whole simulations of one box from a stored state to
their delta power spectra (gev_run_to_outputs), the reference's own call
sequence entry by entry, batches of small boxes, the initial-condition
generator and the power-spectrum estimator.  Cosmology, box sizes (4 or 5
Mpc/h per cell), grids and outputs are those of the library's benchmark,
ensemble and tests.

A simulation changes its box, so a pass first takes the stored initial state
over into the working box (gev_copy_state), as programs do that branch several
runs or both precision forms from one state.

listed()  the cases;  draw(rng)  one more of the same ranges;
prepare(case, seed)  boxes, stored states and tables;  run(state)  one pass;
work(case)  bytes and operations of a pass;  exact(case, seed)  the outputs
in plain numpy where they have such values.
"""
import math
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "gevolution-1.2_amd"))

import bbks  # noqa: E402
import gevpm  # noqa: E402

C_LIGHT = 2997.92458   # 100 km/s units
H_DIM, OMEGA_M, OMEGA_B = 0.67, 0.31, 0.05
Z_IN = 100.0
FORMS = {"fp64": gevpm.FORM_FP64, "fp32": gevpm.FORM_FP32}

# What every kind of case reads from its dict:
#   run      n, form, gr (1 GR, 0 Newton), elliptic (the vector method), cell
#            (Mpc/h), z0 (where the stored state stands), z_pk (texts joined
#            by "/": the outputs), snapshot (return the particles and fields)
#   calls    n, form, cell, z0, cycles: the reference's calls one by one
#   batch    n, form, gr, cell, z0, z_pk, boxes
#   ics      n, cell: initial conditions and their spectrum
#   spectrum n, form: FFT of a field and its power spectrum


def listed():
    return [
        # P(k) of one small field: the shortest call a program makes (two
        # kernels' worth of work, the launch and read-back latency counts)
        {"name": "spectrum-64-fp64", "kind": "spectrum", "n": 64, "form": "fp64"},
        # a small test-sized box run to a snapshot that is taken to the host
        {"name": "run-32-gr-fp64-snapshot", "kind": "run", "n": 32, "form": "fp64", "gr": 1, "elliptic": 0, "cell": 5.0,
         "z0": 100.0, "z_pk": "10", "snapshot": True},
        # a Newtonian comparison run in the precision form, radix-3 grid
        {"name": "run-48-newton-fp32", "kind": "run", "n": 48, "form": "fp32", "gr": 0, "elliptic": 0, "cell": 5.0,
         "z0": 100.0, "z_pk": "0", "snapshot": False},
        # the reference's small configuration in full: z = 100 to 0, three outputs
        {"name": "run-64-gr-fp64-whole", "kind": "run", "n": 64, "form": "fp64", "gr": 1, "elliptic": 0, "cell": 5.0,
         "z0": 100.0, "z_pk": "10/1/0", "snapshot": False},
        # an ensemble of the smallest boxes (parameter studies): one batch
        {"name": "batch-32x48-gr-fp32", "kind": "batch", "n": 32, "form": "fp32", "gr": 1, "cell": 5.0, "z0": 100.0,
         "z_pk": "0", "boxes": 48},
        # a batch of middling boxes, as the serving loop and the ensemble fill them
        {"name": "batch-96x8-gr-fp64", "kind": "batch", "n": 96, "form": "fp64", "gr": 1, "cell": 5.0, "z0": 100.0,
         "z_pk": "10", "boxes": 8},
        # a maintainer who swaps the reference's calls one for one
        {"name": "calls-128-gr-fp64", "kind": "calls", "n": 128, "form": "fp64", "cell": 5.0, "z0": 20.0, "cycles": 8},
        # the start of every program: initial conditions, with their spectrum
        {"name": "ics-192", "kind": "ics", "n": 192, "cell": 5.0},
        # elliptic vector method (T0i projected, three more FFTs), ordinary size
        {"name": "run-192-elliptic-fp64", "kind": "run", "n": 192, "form": "fp64", "gr": 1, "elliptic": 1, "cell": 5.0,
         "z0": 100.0, "z_pk": "30", "snapshot": False},
        # late, clustered cycles in the precision form
        {"name": "run-256-gr-fp32-late", "kind": "run", "n": 256, "form": "fp32", "gr": 1, "elliptic": 0, "cell": 4.0,
         "z0": 1.0, "z_pk": "0", "snapshot": False},
        # late, clustered cycles in FP64 on a large radix-3 grid
        {"name": "run-384-gr-fp64-late", "kind": "run", "n": 384, "form": "fp64", "gr": 1, "elliptic": 0, "cell": 4.0,
         "z0": 0.6, "z_pk": "0.25", "snapshot": False},
        # the headline box (512^3, 2048 Mpc/h) over early cycles: the largest
        {"name": "run-512-gr-fp64", "kind": "run", "n": 512, "form": "fp64", "gr": 1, "elliptic": 0, "cell": 4.0,
         "z0": 100.0, "z_pk": "68", "snapshot": False},
    ]


GRIDS = (16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512)


def draw(rng):
    kind = rng.choice(["run"] * 6 + ["batch"] * 2 + ["calls", "ics", "spectrum"])
    form = rng.choice(["fp64", "fp32"])
    cell = round(rng.uniform(3.0, 6.0), 2)
    if kind == "spectrum":
        return {"kind": kind, "n": rng.choice(GRIDS[2:9]), "form": form, "bins": rng.randint(12, 200)}
    if kind == "ics":
        return {"kind": kind, "n": rng.choice(GRIDS[:9]), "cell": cell}
    if kind == "calls":
        return {"kind": kind, "n": rng.choice(GRIDS[:9]), "form": form, "cell": cell,
                "z0": round(math.exp(rng.uniform(math.log(5.0), math.log(100.0))), 2), "cycles": rng.randint(2, 12)}
    gr = 1 if rng.random() < 0.7 else 0
    # the span in a: a cycle advances ln a by about 0.04
    if kind == "batch":
        n = rng.choice(GRIDS[:7])
        z0 = rng.choice([100.0, 10.0])
        cyc = rng.randint(8, 60)
        boxes = max(2, min(64, int(rng.uniform(0.2, 1.0) * 64 * (32 / n) ** 2)))
        z1 = max(0.0, (1.0 + z0) * math.exp(-0.04 * cyc) - 1.0)
        return {"kind": kind, "n": n, "form": form, "gr": gr, "cell": cell, "z0": z0, "z_pk": "%.2f" % z1, "boxes": boxes}
    n = rng.choice(GRIDS)
    z0 = rng.choice([100.0, 100.0, 10.0, 1.0] if n <= 256 else [100.0, 60.0])
    cyc = rng.randint(2, 6) if n == 512 else rng.randint(3, 12) if n > 256 else rng.randint(4, 60)
    z1 = max(0.0, (1.0 + z0) * math.exp(-0.04 * cyc) - 1.0)
    return {"kind": kind, "n": n, "form": form, "gr": gr, "elliptic": int(gr and rng.random() < 0.2), "cell": cell,
            "z0": z0, "z_pk": "%.2f" % z1, "snapshot": False}


# ---------------------------------------------------------------- set-up

def _sim(n, cell, gr=1, elliptic=0):
    """(SimParams, CycleState at z = 100) of a box of n cells a side (main.cpp:278-295)."""
    size = cell * n
    sim = gevpm.SimParams(gr, elliptic, 48.0, 0.04, Z_IN, 1.5 * size * size / C_LIGHT ** 2,
                          gevpm.make_cosmology(OMEGA_M - OMEGA_B, OMEGA_B, H_DIM))
    a0 = 1.0 / (1.0 + Z_IN)
    return sim, gevpm.CycleState(a0, 0.0, gevpm.next_dtau(sim, n, a0), 0.0, 0.0, 0.0, 0.0, 0, 0)


def _ic_tables(n, cell, seed):
    """generateIC_basic's arguments: crystal template, BBKS table, parameters."""
    size = cell * n
    tpl = gevpm.load_homogeneous_template(os.path.join(ROOT, "tests", "golden", "sc1_crystal.dat"))
    k, d, t = bbks.bbks_table(np.logspace(-5.0, np.log10(300.0), 400), Z_IN, OMEGA_M, H_DIM)
    # (an all-zero generator seed is as good as any other; 32 bits)
    ic = gevpm.ICParams(seed & 0x7FFFFFFF, 1, 1, n // 4, Z_IN, 2.1e-9, 0.965, 0.05, size)
    return ic, tpl, (k * size, d, t * size / H_DIM, d, t * size / H_DIM)


def _copy(st):
    return gevpm.CycleState.from_buffer_copy(st)


def _advance(sim, st, n):
    """The host's part of one cycle (main.cpp:766-874): a, tau, dtau."""
    a = gevpm.rungekutta4bg(st.a, sim.fourpiG, sim.cosmo, 0.5 * st.dtau)
    a = gevpm.rungekutta4bg(a, sim.fourpiG, sim.cosmo, 0.5 * st.dtau)
    st.tau += st.dtau
    st.dtau_old = st.dtau
    st.a = a
    st.dtau = gevpm.next_dtau(sim, n, a)
    st.cycle += 1


def _cycles_to(sim, st, n, z):
    """Cycles after which 1 / a < z + 1 (the cycle that then writes an output at z)."""
    s, c = _copy(st), 0
    while not 1.0 / s.a < z + 1.0:
        _advance(sim, s, n)
        c += 1
    return c


def _stored(case, seed):
    """(stored box, sim, state) at z0: generated initial conditions, evolved
    there; a compact box holds them (one particle set)."""
    n, cell, form = case["n"], case["cell"], FORMS[case["form"]]
    sim, st = _sim(n, cell, case.get("gr", 1), case.get("elliptic", 0))
    ic, tpl, tabs = _ic_tables(n, cell, seed)
    box = gevpm.Box(n, n ** 3, compact=True)
    box.generateIC_basic(sim, ic, tpl, *tabs)
    if form != gevpm.FORM_FP64:
        b32 = gevpm.Box(n, n ** 3, form=form, compact=True)
        b32.copy_state_from(box)
        box.close()
        box = b32
    # the output at z0 lies behind: the stored state is the first one past it
    early = _cycles_to(sim, st, n, case["z0"]) if case["z0"] < Z_IN else 0
    if early:
        box.run_cycles(sim, st, early)
    box.synchronize()
    return box, sim, st


def _zpk(case):
    return [float(z) for z in case["z_pk"].split("/")]


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    s = {"case": case, "kind": kind, "n": n}
    if kind == "spectrum":
        s["box"] = gevpm.Box(n, 0, form=FORMS[case["form"]])
        s["box"].upload_field(gevpm.PHI, _phi(n, seed, case["form"]))
    elif kind == "ics":
        s["box"] = gevpm.Box(n, n ** 3)
        s["sim"], s["st"] = _sim(n, case["cell"])
        s["ic"] = _ic_tables(n, case["cell"], seed)
    elif kind == "batch":
        form = FORMS[case["form"]]
        s["batch"] = gevpm.Batch(n, n ** 3, case["boxes"], gr=case["gr"], form=form)
        # the boxes of a batch differ in their seeds
        s["stored"] = [_stored(case, seed * 1009 + j) for j in range(case["boxes"])]
        s["batch"].autotune()
    else:
        s["stored"] = _stored(case, seed)
        s["box"] = gevpm.Box(n, n ** 3, form=FORMS[case["form"]])
    return s


def _phi(n, seed, form):
    """A potential-like field: of the order of 1e-5, zero mean."""
    phi = 1e-5 * np.random.default_rng(seed).standard_normal((n, n, n))
    return phi.astype(np.float32).astype(np.float64) if form == "fp32" else phi


# ---------------------------------------------------------------- passes

def _tables(out, form):
    """A spectrum table's outputs; the FP32 form's numbers carry float precision."""
    if form == "fp64":
        return dict(out)
    return {k: v.astype(np.float32) if v.dtype == np.float64 and k != "z" else v for k, v in out.items()}


def _spectrum_out(spec, form):
    return _tables(dict(zip(("k", "pk", "sigma_k", "sigma_pk", "occupation"), spec)), form)


def _scalars(st, form):
    """The run's advanced state (phi(k=0) of the FP32 form is a difference of
    rounded sums and stays out)."""
    out = {"a": st.a, "tau": st.tau, "dtau": st.dtau, "cycle": st.cycle}
    if form == "fp64":
        out.update(maxvel=st.maxvel, T00hom=st.T00hom, phi_k0=st.phi_k0)
    else:
        out.update(maxvel=np.float32(st.maxvel), T00hom=np.float32(st.T00hom))
    return out


def run(s):
    return {"spectrum": _run_spectrum, "ics": _run_ics, "batch": _run_batch, "calls": _run_calls,
            "run": _run_box}[s["kind"]](s)


def _run_spectrum(s):
    box, case = s["box"], s["case"]
    box.fft(gevpm.PLAN_PHI, gevpm.FFT_FORWARD)
    return _spectrum_out(box.extractPowerSpectrum(gevpm.SCALARFT, case.get("bins", s["n"] // 2), deconvolve=False),
                         case["form"])


def _delta_spectrum(box, a, n):
    box.projection_init(gevpm.SOURCE)
    box.projection_T00_project(a, True, 1.0)
    box.fft(gevpm.PLAN_SOURCE, gevpm.FFT_FORWARD)
    return box.extractPowerSpectrum(gevpm.SCALARFT, n // 2)


def _run_ics(s):
    ic, tpl, tabs = s["ic"]
    maxvel, disp = s["box"].generateIC_basic(s["sim"], ic, tpl, *tabs)
    out = _spectrum_out(_delta_spectrum(s["box"], s["st"].a, s["n"]), "fp64")
    out.update(maxvel=maxvel, max_displacement=disp)
    return out


def _run_box(s):
    stored, sim, st0 = s["stored"]
    case, box, st = s["case"], s["box"], _copy(st0)
    box.copy_state_from(stored)
    out = _tables(box.run_to_outputs(sim, st, _zpk(case), s["n"] // 2, case["cell"] * s["n"]), case["form"])
    out.update(_scalars(st, case["form"]))
    if case["snapshot"]:
        pos, q, ids = box.download_particles()
        o = np.argsort(ids)
        out.update(pos=pos[o], q=q[o], phi=box.download_field(gevpm.PHI), chi=box.download_field(gevpm.CHI),
                   Bi=box.download_field(gevpm.BI))
    return out


def _run_batch(s):
    case, B = s["case"], s["batch"]
    B.set_outputs(_zpk(case), s["n"] // 2)
    for j, (stored, sim, st) in enumerate(s["stored"]):
        B.box(j).copy_state_from(stored)
        B.start_box(j, sim, st, case["cell"] * s["n"])
    B.run_to_outputs()
    outs = [_tables(B.outputs(j), case["form"]) for j in range(case["boxes"])]
    return {k: np.stack([o[k] for o in outs]) for k in outs[0]}


def _run_calls(s):
    """The main loop of the reference call by call (main.cpp:372-879, GR, parabolic)."""
    stored, sim, st0 = s["stored"]
    case, box, st, N = s["case"], s["box"], _copy(st0), s["n"]
    box.copy_state_from(stored)
    dx, fourpiG, cosmo = 1.0 / N, sim.fourpiG, sim.cosmo
    maxvel, T00 = [], []
    for _ in range(case["cycles"]):
        a = st.a
        box.projection_init(gevpm.SOURCE)
        box.projection_T00_project(a, True, 1.0)
        box.projection_init(gevpm.SIJ)
        box.projection_Tij_project(a, True, 1.0)
        T00.append(box.field_sum(gevpm.SOURCE) / N ** 3)
        if st.dtau_old > 0.0:
            H = gevpm.hconf(a, fourpiG, cosmo)
            box.prepareFTsource_scalar(cosmo.Omega_cdm + cosmo.Omega_b, 3.0 * H * dx * dx / st.dtau_old,
                                       fourpiG * dx * dx / a, 3.0 * H * H * dx * dx)
            box.fft(gevpm.PLAN_SOURCE, gevpm.FFT_FORWARD)
            box.solveModifiedPoissonFT(1.0 / (dx * dx), 3.0 * H / st.dtau_old)
            box.fft(gevpm.PLAN_PHI, gevpm.FFT_BACKWARD)
        box.prepareFTsource_tensor(2.0 * fourpiG * dx * dx / a)
        box.fft(gevpm.PLAN_SIJ, gevpm.FFT_FORWARD)
        box.projectFTscalar()
        box.fft(gevpm.PLAN_CHI, gevpm.FFT_BACKWARD)
        box.evolveFTvector(a * a * st.dtau_old)
        box.fft(gevpm.PLAN_BI, gevpm.FFT_BACKWARD)
        nfk = 3 if 1.0 / a < sim.z_relax + 1.0 else 2
        maxvel.append(box.updateVel(gevpm.Q_GR, 0.5 * (st.dtau + st.dtau_old), nfk, [a, a * a * N]))
        a = gevpm.rungekutta4bg(a, fourpiG, cosmo, 0.5 * st.dtau)
        nfd = 3 if 1.0 / a < sim.z_relax + 1.0 else 0
        box.moveParticles(gevpm.POS_GR, st.dtau, nfd, [a, a * a * N])
        _advance(sim, st, N)
    out = _spectrum_out(_delta_spectrum(box, st.a, N), case["form"])
    t = np.float64 if case["form"] == "fp64" else np.float32
    out.update(maxvel=np.array(maxvel, dtype=t), T00hom=np.array(T00, dtype=t), a=st.a)
    return out


# ---------------------------------------------------------------- work

def _cycle_work(n, f, gr, elliptic):
    """Bytes and operations of one cycle (f: bytes of a real field element):
    every carried field and particle array read once and written once by each
    stage that has to materialise it, the FFT chains as one read of their
    inputs and one write of their outputs; an FFT as 2.5 n^3 log2(n^3)."""
    c, k = n ** 3, n * n * (n // 2 + 1) * 2 * f
    by = 48 * c + f * c + 7 * f * c          # deposit: pos, q, phi in; T00 + Tij out
    by += f * c + 3 * f * c + f * c          # T00hom; phi, chi, source in, phi out
    by += 7 * f * c + 6 * k + 4 * f * c      # phi, Tij and BiFT in; BiFT, chi and B out
    by += 96 * c + 5 * f * c                 # kick and drift
    by += 8 * c + 4 * c + 8 * c + 12 * c     # cells, counts, offsets, permutation
    ffts = 12 if gr else 9
    if elliptic:
        by += 48 * c + 6 * f * c + 3 * k
        ffts += 3
    return by, ffts * 2.5 * c * math.log2(c) + c * (8 * 60 + 400) + 0.5 * c * 300


def work(case):
    n, kind = case["n"], case["kind"]
    f = 4 if case.get("form") == "fp32" else 8
    c = n ** 3
    spec_b, spec_f = f * c, 2.5 * c * math.log2(c) + 20 * c    # a field's transform and its bins
    delta_b, delta_f = 48 * c + 2 * f * c + spec_b, spec_f + 8 * 15 * c
    if kind == "spectrum":
        return {"bytes": spec_b, "flops": spec_f}
    if kind == "ics":
        # three realisations, 15 transforms, two deposits, displacement and momenta
        return {"bytes": 15 * 8 * c + 2 * 48 * c + 9 * 8 * c + 104 * c + 11 * 8 * c + delta_b,
                "flops": 15 * 2.5 * c * math.log2(c) + 600 * c + delta_f}
    sim, st = _sim(n, case["cell"], case.get("gr", 1), case.get("elliptic", 0))
    for _ in range(_cycles_to(sim, st, n, case["z0"]) if case["z0"] < Z_IN else 0):
        _advance(sim, st, n)
    by, fl = _cycle_work(n, f, case.get("gr", 1), case.get("elliptic", 0))
    # the stored state taken over: particles, the carried fields, the filing
    over = 2 * (56 * c + 5 * f * c + 3 * 2 * f * n * n * (n // 2 + 1)) + 24 * c
    if kind == "calls":
        return {"bytes": case["cycles"] * by + over + delta_b, "flops": case["cycles"] * fl + delta_f}
    z = _zpk(case)
    cycles = max(1, _cycles_to(sim, st, n, z[-1]))
    m = case.get("boxes", 1)
    # an output is written twice (the look-ahead write and the interpolated one)
    return {"bytes": m * (cycles * by + over + 2 * len(z) * delta_b), "flops": m * (cycles * fl + 2 * len(z) * delta_f)}


# ---------------------------------------------------------------- exact values

def exact(case, seed):
    """The spectrum cases in numpy: rfftn and the estimator of tools.hpp:53-212
    (power weighted by k^3, linear k, not deconvolved).  The simulations have
    no such values in reach."""
    if case["kind"] != "spectrum" or case["n"] > 192:
        return None
    n, h, bins = case["n"], case["n"] // 2, case.get("bins", case["n"] // 2)
    F = np.fft.rfftn(_phi(n, seed, case["form"]))
    i = np.arange(n)
    tk = (2.0 * np.pi * np.minimum(i, n - i)) ** 2
    k2 = (tk[None, None, :h + 1] + tk[None, :, None]) + tk[:, None, None]
    w = np.broadcast_to(np.where((i[:h + 1] == 0) | (i[:h + 1] == h), 1.0, 2.0), k2.shape)
    b = np.floor(bins * np.sqrt(k2 / (3.0 * tk[h]))).astype(np.int64)
    live = b < bins
    live[0, 0, 0] = False
    b, w, kk = b[live], w[live], np.sqrt(k2[live])
    p = np.abs(F[live]) ** 2 * kk ** 3
    occ = np.bincount(b, weights=w, minlength=bins)
    some = np.maximum(occ, 1.0)
    kbin = np.bincount(b, weights=w * kk, minlength=bins) / some
    power = np.bincount(b, weights=w * p, minlength=bins) / some
    return {"k": kbin, "pk": power, "sigma_k": None, "sigma_pk": None, "occupation": None}
