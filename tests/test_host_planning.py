"""CPU tests of the host side that plans a step (kaminogpu_amd/csrc/
kamino_runtime.hip): a small C++ program linked with the library calls it, with
no GPU call made."""
import math
import os
import shutil
import subprocess

import numpy as np
import pytest

import kaminogpu_amd as K

PKG = os.path.dirname(os.path.abspath(K.__file__))
ROOT = os.path.dirname(PKG)

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")


def run_cpp(tmp_path, source, *args):
    """Builds `source` against the library and returns what it prints."""
    K.lib()
    src, exe = tmp_path / "main.cpp", tmp_path / "main"
    src.write_text(source)
    build = ["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"),
             "-I", os.path.join(PKG, "csrc"), "-isystem", "/opt/rocm/include", "-o", str(exe), str(src),
             "-pthread", "-L", PKG, "-lkamino", f"-Wl,-rpath,{PKG}", "-Wl,-rpath-link,/opt/rocm/lib"]
    r = subprocess.run(build, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-2000:])
    return r.stdout


# Every heap allocation of the process goes through these; the no-allocation
# step (kam_sim_step_noalloc) plans its shape and fills its tables on the host.
COUNTED = r"""
#include <cstdio>
#include <cstdlib>
#include <new>

#include "kamino.h"
#include "kamino_runtime.h"

static long g_count = 0;
void* operator new(std::size_t n) {
    ++g_count;
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

static float rowf[kam::RT_COUNT * 512], tw[4 * 512];
static double rowd[kam::RD_COUNT * 512], tw64[4 * 512];

int main() {
    long plans = 0;
    for (int pass = 0; pass < 2; ++pass)
        for (int n = 4; n <= 512; ++n) {
            int m = n;
            for (int p : {2, 3, 5})
                while (m % p == 0) m /= p;
            if (m != 1) continue;
            kam::Plan plan;
            const long before = g_count;
            if (kam::make_plan(n, 2 * n, plan) != KAM_OK) return 1;
            if (pass) kam::compute_tables(n, 0.5 / n, 1.0, rowf, rowd, tw, tw64);
            if (g_count != before) std::printf("n_theta %d: %ld allocations\n", n, g_count - before);
            ++plans;
        }
    std::printf("%ld plans\n", plans);
    return 0;
}
"""


def test_planning_a_shape_uses_no_heap(tmp_path):
    sizes = [n for n in range(4, 513) if (2 * 3 * 5) ** 9 % n == 0]  # 2^a 3^b 5^c
    assert run_cpp(tmp_path, COUNTED) == f"{2 * len(sizes)} plans\n"


# Eight threads plan every size at once, each in its own order.
THREADS = r"""
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

#include "kamino_runtime.h"

int main() {
    std::vector<int> sizes;
    for (int n = 4; n <= kam::kMaxTheta; ++n) {
        int m = n;
        for (int p : {2, 3, 5})
            while (m % p == 0) m /= p;
        if (m == 1) sizes.push_back(n);
    }
    std::atomic<int> ready{0}, bad{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([&, t] {
            ++ready;
            while (ready < 8) {}
            for (size_t k = 0; k < sizes.size(); ++k) {
                const int n = sizes[t & 1 ? sizes.size() - 1 - k : k];
                kam::Plan p;
                if (kam::make_plan(n, 2 * n, p) != KAM_OK) {
                    ++bad;
                    continue;
                }
                // complete: the passes' radices multiply to M (their items, to M / R)
                const kam::FftPlan& f = p.size->fft;
                long left = n;
                for (int q = 0; q < f.nPass; ++q) left /= n / f.pass[q].nb;
                if (left != 1 || f.lanes < 8 || !(p.size->sinPole > 0.0)) ++bad;
            }
        });
    for (auto& t : threads) t.join();
    std::printf("%zu sizes, %d bad\n", sizes.size(), bad.load());
    return 0;
}
"""


def test_planning_from_several_threads(tmp_path):
    assert run_cpp(tmp_path, THREADS) == "107 sizes, 0 bad\n"


# Tiles of one sphere's particles, from `plan_tiles` alone.
PARTICLES = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "kamino_runtime.h"

int main(int, char** argv) {
    const int nT = std::atoi(argv[1]);
    const long long n = std::atoll(argv[2]);
    kam::Plan plan;
    if (kam::make_plan(nT, 2 * nT, plan) != KAM_OK) return 1;
    kam_sim_desc sd{};
    sd.n_theta = nT;
    sd.n_phi = 2 * nT;
    sd.radius = 1.0;
    sd.dt = 0.5 / nT;
    sd.geometric = 1;
    kam::SimDesc d;
    kam::fill_desc(d, plan, kam::Tables(), sd, nullptr);
    d.nPart = (int)n;
    int rows[4];
    kam::TileLayout L;
    const int need = kam::plan_tiles(&d, &plan, 1, rows, nullptr, 0, L);
    std::vector<kam::Tile> tiles((size_t)need);
    kam::plan_tiles(&d, &plan, 1, rows, tiles.data(), need, L);
    long long next = 0;  // the tiles cover every particle once, in order
    int longest = 0;
    for (int t = 0; t < L.nPart; ++t) {
        const kam::Tile& tile = tiles[(size_t)(L.partOff + t)];
        if (tile.row0 != next || tile.rows < 1) return 2;
        next += tile.rows;
        longest = std::max(longest, tile.rows);
    }
    if (next != n) return 3;
    std::printf("%d %d %d\n", L.nPartLds, L.nPart, longest);
    return 0;
}
"""


def test_particle_tiles_are_few(tmp_path):
    """A tile is 16 bytes to plan, stage and upload for at least 2048 particles."""
    for nt, n in [(32, 1), (64, 2048), (64, 2049), (128, 100_000), (256, 1_000_000), (64, 1 << 26)]:
        sub = tmp_path / f"{nt}_{n}"
        sub.mkdir()
        staged, tiles, longest = map(int, run_cpp(sub, PARTICLES, str(nt), str(n)).split())
        assert staged == 0 and tiles == -(-n // 2048) and longest <= 2048, (nt, n, staged, tiles, longest)


# The autotuner's choice; arguments: rounds, then the times of each round.
PICK = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "kamino_runtime.h"

int main(int argc, char** argv) {
    const int rounds = std::atoi(argv[1]);
    std::vector<double> ms;
    for (int k = 2; k < argc; ++k) ms.push_back(std::atof(argv[k]));
    std::printf("%d\n", kam::pick_shape(ms.data(), rounds, (int)ms.size() / rounds));
    return 0;
}
"""


def test_autotuner_keeps_the_default_among_equals(tmp_path):
    """Clocks that rise through the timings make later shapes look faster, and
    equal shapes differ by some percent: neither moves the choice, nor does one
    round that runs off.  A shape that is clearly faster does, of several the
    fastest, or the first of those that time alike."""
    rng = np.random.default_rng(3)

    def pick(name, rel, noise=0.02, drift=0.0):
        ms = np.empty((5, len(rel)))
        for t, i in enumerate(np.ndindex(ms.shape)):
            ms[i] = rel[i[1]] * (1 + drift * math.exp(-t / 4)) * (1 + noise * rng.uniform(-1, 1))
        sub = tmp_path / name
        sub.mkdir()
        return int(run_cpp(sub, PICK, "5", *(f"{x:.6f}" for x in ms.ravel())))

    for k in range(6):
        assert pick(f"equal{k}", [1.0] * 9, drift=0.3) == 0
    assert pick("faster", [1.0, 1.02, 0.9, 0.85, 0.99], drift=0.3) == 3
    assert pick("alike", [1.0, 1.02, 0.90, 0.895, 0.89], noise=0.005) == 2
    assert pick("slower", [1.0, 1.2, 1.1]) == 0
    sub = tmp_path / "once"
    sub.mkdir()
    assert int(run_cpp(sub, PICK, "3", *"1 0.99 0.8 1 0.98 0.8 1.5 0.98 0.85".split())) == 2
    assert int(run_cpp(sub, PICK, "3", *"1 0.99 1 0.98 1.5 0.98".split())) == 0


def test_fft_heights_a_tuning_entry_may_name():
    """Heights up to (20480 complex values of LDS) / M less three rows and a row
    per lane group are taken, as many rows as the sphere has at most; taller
    ones leave the default.  At 256 rows LDS holds one row less than the limit."""
    for nt in [n for n in range(4, 2049) if (2 * 3 * 5) ** 11 % n == 0]:
        K.tune_set(nt, 0, 0, 0)
        default = K.tune_get(nt)[2]
        lanes = next((g for g in (8, 16, 32) if 4 * g >= nt), 64) if nt < 1024 else 256
        limit = 20480 // nt - 3 - 256 // lanes
        try:
            for rows in (1, 2, limit - 1, limit, limit + 1, 10 ** 6):
                K.tune_set(nt, 0, 0, rows)
                want = min(rows, nt, 72 if nt == 256 else nt) if rows <= limit else default
                assert K.tune_get(nt)[2] == want, (nt, rows, limit)
        finally:
            K.tune_set(nt, 0, 0, 0)
