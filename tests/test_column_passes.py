"""The strided FFT passes' tiles (csrc/fft_core.h), with the header's own rules
compiled on the host: for every compiled grid size, form, axis and row width
the workgroups take every column once, the 32-bit byte offset of a thread
holds, the tile fits a workgroup and its LDS, and the register stages
(ColumnTile), restated in numpy job by job with their masks, transform a tile
as numpy does, reading and writing every element once.  CPU only."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from test_index_bounds import SIZES, kpitch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gevolution-1.2_amd", "csrc")
TSV = os.path.join(ROOT, "gevolution-1.2_amd", "lib", "kernel_resources.tsv")
HIPCC = os.environ.get("HIPCC") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc"))

SOURCE = r"""
#include <cstdio>
#include "fft_core.h"
using namespace gev_fft;
template <typename T, int N, int RB> void row(int elem) {
    printf("%d %d %d %d %d %d\n", elem, N, RB, col_tile<T, N, RB>(), col_tpb<T, N, RB>(), x_lines<N>());
}
template <typename T, int N> void size(int elem) {
    row<T, N, 0>(elem);
    if (N <= 256) row<T, N, 64>(elem), row<T, N, 256>(elem);
}
template <int N> void both() { size<double, N>(8), size<float, N>(4); }
template <int... N> void all() { (both<N>(), ...); }
int main() { all<SIZES>(); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """{(element bytes, N, row bytes asked for): (columns, threads, x lines)}"""
    if not HIPCC:
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("rules")
    src, exe = str(d / "rules.cpp"), str(d / "rules")
    with open(src, "w") as f:
        f.write(SOURCE.replace("SIZES", ", ".join(map(str, SIZES))))
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I", CSRC, src,
                    "-o", exe], check=True, capture_output=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    r = {}
    for line in out.split("\n"):
        if line:
            e, n, rb, w, t, x = map(int, line.split())
            r[e, n, rb] = (w, t, x)
    return r


def radix(n):
    return 8 if n % 8 == 0 else 4 if n % 4 == 0 else 2 if n % 2 == 0 else 3


def test_rules_are_of_every_size(rules):
    assert len(rules) == 2 * (len(SIZES) + 2 * sum(n <= 256 for n in SIZES))


def test_tiles_fit_and_cover(rules):
    for (elem, N, rb), (W, NT, _) in rules.items():
        c, H, P = 2 * elem, N // 2 + 1, kpitch(N)
        assert NT % 64 == 0 and 64 <= NT <= 1024 and NT % W == 0, (elem, N, rb)
        assert (N * W + N) * c <= 160 * 1024, (elem, N, rb)  # tile and twiddles
        # the rows a thread reaches from its own (ev) stay below a 32-bit byte offset, y and z passes
        for es in (P, P * N):
            assert ((NT // W - 1) * es + W - 1) * c < 2 ** 32, (elem, N, rb)
        ntx = (H + W - 1) // W
        grid = ntx * N
        l = np.arange(grid)
        if grid % 8 == 0:
            l = l % 8 * (grid // 8) + l // 8
        assert len(np.unique(l)) == grid and l.max() < grid, (elem, N, rb)
        assert (l // ntx).max() == N - 1
        cols = np.add.outer(l % ntx * W, np.arange(W))
        assert sorted(set(cols[l // ntx == 0].ravel()) & set(range(H))) == list(range(H))


def stage_of(x, N, W, R, NS, jobs, twiddled=True):
    """Operands, results and their elements of one stage's jobs."""
    M = N // R
    w, j = jobs % W, jobs // W
    k = j % NS
    e = j[:, None] + np.arange(R) * M
    v = x[e, w[:, None]]
    if twiddled:
        v = v * np.exp(-2j * np.pi * (k[:, None] * np.arange(R) * (N // (NS * R))) / N)
    v = np.fft.fft(v, axis=1)
    return e, (j // NS * NS * R + k)[:, None] + np.arange(R) * NS, w, v


@pytest.mark.parametrize("N", SIZES)
def test_register_stages_transform_a_tile(rules, N):
    rng = np.random.default_rng(N)
    for (elem, n, rb), (W, NT, _) in rules.items():
        if n != N:
            continue
        x = rng.standard_normal((N, W)) + 1j * rng.standard_normal((N, W))
        want = np.fft.fft(x, axis=0)
        R1 = radix(N)
        # first stage: butterfly t of thread tid is job tid + t NT, loaded as
        # element ev + t (NT / W) + r N / R1 of its column (masked past the jobs)
        M1, njobs = N // R1, W * (N // R1)
        tid = np.arange(NT)
        lds = np.full((N, W), np.nan, dtype=complex)
        seen = np.zeros((N, W), dtype=int)
        for t in range((njobs + NT - 1) // NT):
            on = tid + t * NT < njobs
            jobs = (tid + t * NT)[on]
            e = (tid // W)[on][:, None] + t * (NT // W) + np.arange(R1) * M1
            assert e.max() < N
            np.add.at(seen, (e, (tid % W)[on][:, None]), 1)
            assert np.array_equal(e, (jobs // W)[:, None] + np.arange(R1) * M1)
            _, d, w, v = stage_of(x, N, W, R1, 1, jobs, False)
            if R1 == N:  # a single stage stores from the registers
                d = (tid // W)[on][:, None] + t * (NT // W) + np.arange(R1) * M1
            lds[d, w[:, None]] = v
        assert (seen == 1).all(), (elem, rb)
        NS = R1
        while NS < N:
            R = radix(N // NS)
            jobs = np.arange(W * (N // R))
            e, d, w, v = stage_of(lds, N, W, R, NS, jobs)
            if NS * R == N:
                # the last stage stores element ev + t (NT / W) + r NS, masked past the jobs
                out = np.full((N, W), np.nan, dtype=complex)
                seen = np.zeros((N, W), dtype=int)
                for t in range((len(jobs) + NT - 1) // NT):
                    on = tid + t * NT < len(jobs)
                    el = (tid // W)[on][:, None] + t * (NT // W) + np.arange(R) * NS
                    assert el.max() < N
                    jj = (tid + t * NT)[on]
                    out[el, (tid % W)[on][:, None]] = v[jj]
                    np.add.at(seen, (el, (tid % W)[on][:, None]), 1)
                assert (seen == 1).all(), (elem, rb)
                lds = out
            else:
                nxt = np.full((N, W), np.nan, dtype=complex)
                nxt[d, w[:, None]] = v
                lds = nxt
            NS *= R
        assert np.allclose(lds, want, rtol=0, atol=1e-12 * N), (elem, rb)


def test_x_rows(rules):
    """The x passes' rows per workgroup: all rows taken, LDS of padded lines within 64 KiB."""
    for (elem, N, rb), (_, _, lines) in rules.items():
        M = N // 2
        assert lines >= 1 and lines * M <= (512 if N <= 128 else 2048)
        assert lines * (M + M // 16) * 2 * elem + M * 2 * elem <= 64 * 1024
        assert (N * N + lines - 1) // lines * lines >= N * N


@pytest.mark.parametrize("mangled,waves", [
    ("k_c2c_colsIdLi768E", 3),  # one butterfly per thread; 2 with two each, which took 1.63 ms for the 1.55 of a y pass
    ("k_c2c_colsIfLi768E", 6),  # 3 with two each (1.02 ms, 0.78)
    ("k_c2c_colsIfLi384E", 6),
])
def test_wavefronts_of_the_radix_3_sizes(mangled, waves):
    if not os.path.exists(TSV):
        pytest.skip("library not built with its resource report")
    import csv
    with open(TSV) as f:
        occ = [int(r["occupancy"]) for r in csv.DictReader(f, delimiter="\t") if mangled in r["kernel"]]
    assert occ and min(occ) >= waves, occ
