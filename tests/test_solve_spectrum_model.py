"""Host model of the tensor z pass that solves on registers (k_zsolve_direct),
of the tensor x pass's row rules and of the spectrum's row kernel, which
tests/test_index_bounds.py predates: the solve restated thread by thread in
numpy (loads, stages, the halves that the two groups trade, stores), the row
counts, the run list, and the LDS of the spectrum against the compiler's
report.  CPU only."""
import csv
import os
import re

import numpy as np
import pytest

from test_index_bounds import CSRC, SIZES, kpitch

TSV = os.path.join(os.path.dirname(CSRC), "lib", "kernel_resources.tsv")


def source(name):
    with open(os.path.join(CSRC, name)) as f:
        return f.read()


def number(name, pattern):
    m = re.search(pattern, source(name))
    assert m, pattern
    return int(m.group(1))


@pytest.fixture(scope="module")
def rows():
    if not os.path.exists(TSV):
        pytest.skip("library not built with its resource report")
    with open(TSV) as f:
        return list(csv.DictReader(f, delimiter="\t"))


# ---------------------------------------------------------------- k_zsolve_direct

W = number("fftsolve.hip", r"constexpr int ZD_COLS = (\d+);")
DIRECT = (64, 128, 256, 512)


def test_the_model_knows_which_sizes_are_direct():
    assert "KIND == ZS_TENSOR && N >= 64 && N <= 512 && (N & (N - 1)) == 0" in source("fftsolve.hip")


def radix(n):
    return 8 if n % 8 == 0 else 4 if n % 4 == 0 else 2


def transform(v, N):
    """zd_transform of one group: v[T][8], point m of thread (ev, w) is element
    ev + m N / 8 of column w; the same layout comes back."""
    T = len(v)
    ev, w = np.arange(T) // W, np.arange(T) % W
    buf = np.full(N * W, np.nan, dtype=complex)
    x = np.fft.fft(v, axis=1)
    for r in range(8):
        buf[(ev * 8 + r) * W + w] = x[:, r]
    NS = 8
    while True:
        R = radix(N // NS)
        J = 8 // R
        out, nxt = np.empty((T, 8), dtype=complex), np.full(N * W, np.nan, dtype=complex)
        for t in range(J):
            j = ev + t * (N // 8)
            k = j % NS
            assert (j + (R - 1) * (N // R)).max() < N
            u = np.stack([buf[(j + r * (N // R)) * W + w] for r in range(R)], axis=1)
            u = np.fft.fft(u * np.exp(-2j * np.pi * k[:, None] * np.arange(R) / (NS * R)), axis=1)
            for r in range(R):
                out[:, t + r * J] = u[:, r]
                nxt[(j // NS * NS * R + k + r * NS) * W + w] = u[:, r]
        NS *= R
        if NS == N:
            return out
        buf = nxt


@pytest.mark.parametrize("N", DIRECT)
def test_direct_solve_moves_every_point_once(N):
    T = N * W // 8
    rng = np.random.default_rng(N)
    f = rng.standard_normal((6, N, W)) + 1j * rng.standard_normal((6, N, W))
    ev, w = np.arange(T) // W, np.arange(T) % W
    own = [np.stack([f[c][ev + m * (N // 8), w] for m in range(8)], axis=1) for c in range(6)]
    F = np.fft.fft(f, axis=1)
    S = np.empty((2, 6, T, 4), dtype=complex)  # by group
    for r in range(3):
        X = [transform(own[2 * r + g], N) for g in (0, 1)]
        s_x = np.full(N * W, np.nan, dtype=complex)
        for g in (0, 1):
            for i in range(4):
                s_x[(g * 4 + i) * T + np.arange(T)] = X[g][:, i] if g else X[g][:, 4 + i]
        for g in (0, 1):
            for i in range(4):
                other, mine = s_x[((1 - g) * 4 + i) * T + np.arange(T)], X[g][:, 4 + i] if g else X[g][:, i]
                S[g, 2 * r, :, i], S[g, 2 * r + 1, :, i] = (other, mine) if g else (mine, other)
    seen = np.zeros((N, W), dtype=int)
    for g in (0, 1):
        for i in range(4):
            kz = ev + (4 * g + i) * (N // 8)
            np.add.at(seen, (kz, w), 1)
            for c in range(6):
                assert np.allclose(S[g, c, :, i], F[c][kz, w], rtol=0, atol=1e-11 * N), (g, c, i)
    assert (seen == 1).all()
    O = S[:, :4]  # any function of the point; here the first four components
    for r in range(2):
        oa, ob = 2 * r, 2 * r + 1
        s_x = np.full(N * W, np.nan, dtype=complex)
        for g in (0, 1):
            for i in range(4):
                s_x[(g * 4 + i) * T + np.arange(T)] = O[g, oa, :, i] if g else O[g, ob, :, i]
        for g in (0, 1):
            v = np.empty((T, 8), dtype=complex)
            for i in range(4):
                other, mine = s_x[((1 - g) * 4 + i) * T + np.arange(T)], O[g, ob, :, i] if g else O[g, oa, :, i]
                v[:, i], v[:, 4 + i] = (other, mine) if g else (mine, other)
            back = np.conj(transform(np.conj(v), N)) / N
            for m in range(8):
                assert np.allclose(back[:, m], f[oa + g][ev + m * (N // 8), w], rtol=0, atol=1e-11 * N), (r, g, m)


@pytest.mark.parametrize("N", DIRECT)
def test_direct_solve_in_bounds(N):
    P, H = kpitch(N), N // 2 + 1
    nk, es, T = P * N * N, P * N, N * W // 8
    assert 2 * T <= 1024 and (T - 1) // W == N // 8 - 1
    assert ((N // 8 - 1) * es + W - 1) * 16 < 2 ** 32
    ntx = (H + W - 1) // W
    l = np.arange(ntx * N)
    if len(l) % 8 == 0:
        l = l % 8 * (len(l) // 8) + l // 8
    assert len(np.unique(l)) == len(l) and l.max() < len(l)
    # the last point of the last column within H (columns beyond are masked)
    assert 5 * nk + (N - 1) * P + (H - 1) + 7 * es * (N // 8) + (N // 8 - 1) * es < 6 * nk
    assert (2 * N * W + N * W + N) * 16 <= 160 * 1024


@pytest.mark.parametrize("N", DIRECT)
def test_direct_solve_occupancy(rows, N):
    """The registers of 8 points of the tensor's components leave two waves per
    SIMD (the limit that the workgroup's LDS sets at 512^3 as well)."""
    occ = [int(r["occupancy"]) for r in rows if "k_zsolve_directILi%dE" % N in r["kernel"]]
    assert len(occ) == 1 and occ[0] >= 2, occ


def test_general_tensor_solve_occupancy(rows):
    """The general tensor solve keeps two waves per SIMD at every size it runs."""
    for N in SIZES:
        for elem in "df":
            occ = [int(r["occupancy"]) for r in rows
                   if re.search(r"k_zsolveILi%dELi1E15HIP_vector_typeI%s" % (N, elem), r["kernel"])]
            assert len(occ) == (0 if elem == "d" and N in DIRECT else 1) and all(o >= 2 for o in occ), (N, elem, occ)


# ---------------------------------------------------------------- tensor x pass

PTS = number("fftsolve.hip", r"#define GEV_XPREP_PTS (\d+)")


def x_lines(N):
    m, l = N // 2, 1
    while l * 2 * m <= (512 if N <= 128 else 2048):
        l *= 2
    return l


@pytest.mark.parametrize("N", SIZES)
def test_prepared_rows(N):
    """Rows per workgroup of the scalar, the six-component (over up to twice
    the rows too) and the one-component form: the registers a thread holds,
    the LDS of the padded lines, and every row taken."""
    M = N // 2
    six = x_lines(N)
    while six > 1 and six * M > PTS * 256:
        six //= 2
    one = x_lines(N)
    while one > 1 and one * M > 512:
        one //= 2
    wide = x_lines(N)
    while wide * N <= 2048:
        wide *= 2
    while wide > 1 and wide * M > PTS * 256:
        wide //= 2
    assert six <= wide <= 4 * six and wide * M <= 1024
    for lines in (x_lines(N), six, wide, one):
        assert lines >= 1 and -(-N * N // lines) * lines >= N * N
        assert (lines * (M + M // 16) + M) * 16 <= 64 * 1024
    assert six * M <= PTS * 256 and (one * M <= 512 or one == 1)


# ---------------------------------------------------------------- spectrum

LONG = {385: (4, 2), 513: (4, 2)}
INSTANCES = {65: (4,), 257: (4,), **LONG}


def maxh_of(N):
    return min(h for h in INSTANCES if N // 2 + 1 <= h)


def test_spectrum_lds(rows):
    """Two workgroups fit a CU's 160 KiB at every grid size and bin count (with
    one, a 768^3 spectrum of 384 bins took 7.6 ms for the 4.2 of two)."""
    static = {}
    for r in rows:
        m = re.search(r"k_spectrum_rowsILi(\d+)ELi(\d+)E", r["kernel"])
        if m:
            static.setdefault((int(m.group(1)), int(m.group(2))), set()).add(int(r["lds"]))
    assert sorted(static) == sorted((h, n) for h, ns in INSTANCES.items() for n in ns)
    for N in SIZES:
        h = maxh_of(N)
        four = 4 * h * (3 * 8 + 2 * 2) + h * 8 + 256
        if h in LONG:
            assert four >= max(static[h, 4])  # what the rule counts covers the kernel's own
        for bins in range(1, 1025):
            shm = 36 * bins
            rows_at_once = 2 if h in LONG and four + shm > 80 * 1024 else 4
            assert 2 * (max(static[h, rows_at_once]) + shm) <= 160 * 1024, (N, bins)


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("bins", (1, 7, 64, 1024))
def test_run_list(N, bins):
    """Runs of a row listed 64 modes at a time (the last lane's bin carried
    over): at most H + 1 of them, their ends where the next begins, the last
    at H + 1; no two inside the bins share a bin."""
    H = N // 2
    t = (2.0 * np.pi * np.minimum(np.arange(N), N - np.arange(N))) ** 2
    for ky, kz in ((0, 0), (1, 0), (H, H), (N // 3, N - 1)):
        b = np.floor(bins * np.sqrt((t[:H + 1] + t[ky] + t[kz]) / (3.0 * t[H]))).astype(int)
        b = np.where(b < bins, b, -1)
        if ky == kz == 0:
            b[0] = -1
        run, last = [], -2
        for kb in range(0, H + 1, 64):
            lane = np.arange(64)
            bin_ = np.where(kb + lane <= H, b[np.minimum(kb + lane, H)], -1)
            up = np.concatenate([[last], bin_[:-1]])
            run += [kb + int(l) for l in lane[(kb + lane <= H) & (bin_ != up)]]
            last = bin_[63]
        assert len(run) <= H + 1 <= maxh_of(N)
        ends = run[1:] + [H + 1]
        assert run[0] == 0 and all(len(set(b[s:e])) == 1 for s, e in zip(run, ends))
        inside = [b[s] for s in run if b[s] >= 0]
        assert len(inside) == len(set(inside))
