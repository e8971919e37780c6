"""Work-item depths of a batch (csrc/ttsh_layout.h) on the CPU: over random
batches the depth of the least predicted time is the one that a search over
every droplet and every depth finds, and the search takes no more tile counts
than sizes times the depths that split one of them differently, however many
droplets there are.  And the K_rhs variant that a droplet runs: never one that
its size does not fit."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bacterial-droplet_amd", "csrc")

DRIVER = r"""
#include "ttsh_layout.h"
#include <cstdio>
#include <random>
using namespace ttsh;

static long g_calls = 0;
static int tiles60(int n) { ++g_calls; return ((n + 59) / 60) * ((n + 15) / 16); }
static int tiles32(int n) { ++g_calls; return ((n + 31) / 32) * ((n + 7) / 8); }
static int tiles62(int n) { ++g_calls; return ((n + 61) / 62) * ((n + 13) / 14); }

struct Droplet { int N, ptz; };

static double plain_time(const std::vector<Droplet>& ds, int d, double over, double at_once, int (*tiles)(int))
{
    double items = 0, deepest = 0;
    for (auto& s : ds) {
        const int nz = (s.N + d - 1) / d;
        items += (double)tiles(s.N) * nz;
        deepest = std::max(deepest, (double)((s.N + nz - 1) / nz));
    }
    const double r = items / at_once;
    return (r < 3 ? std::ceil(r) : r + 0.5) * (deepest + over);
}

int main()
{
    const int grid[22] = {32, 36, 40, 48, 50, 60, 64, 72, 80, 90, 96, 100, 120, 128, 144, 150, 160, 180, 192, 200, 240, 256};
    std::mt19937 rng(3);
    for (int trial = 0; trial < 400; ++trial) {
        const int n = 2 + (int)(rng() % (trial % 10 == 9 ? 2000 : 30)), hi = 4 + (int)(rng() % 19);
        std::vector<Droplet> ds;
        std::vector<SizeCount> sizes;
        int N = 0;
        for (int k = 0; k < n; ++k) {
            const Droplet d{grid[rng() % std::min(hi, 22)], 2 + (int)(rng() % 3) * 7};
            ds.push_back(d);
            count_size(sizes, d.N, d.ptz);
            N = std::max(N, d.N);
        }
        int total = 0;
        for (auto& s : sizes) total += s.n;
        if (total != n || sizes.size() > 66) return 1;
        const auto depths = chunk_depths(sizes, N);
        for (double at_once : {256.0, 1024.0})
            for (auto tiles : {tiles60, tiles32}) {
                g_calls = 0;
                const Depth got = least_depth(sizes, depths, 3.0, at_once, tiles);
                if (g_calls > (long)(sizes.size() * depths.size())) return 2;
                int want = 1;
                for (int d = 2; d <= N; ++d)
                    if (plain_time(ds, d, 3.0, at_once, tiles) < plain_time(ds, want, 3.0, at_once, tiles)) want = d;
                if (got.d != want || got.time != plain_time(ds, want, 3.0, at_once, tiles)) {
                    std::printf("depth %d, searched %d\n", got.d, want);
                    return 3;
                }
            }
        // the divergence: the same time as over every droplet
        g_calls = 0;
        const int dd = div_depth(sizes, N, 256, tiles62);
        if (g_calls > (long)sizes.size() * N) return 4;
        double best = 0, mine = 0;
        for (int d = 1; d <= N; ++d) {
            double all = 0, longest = 0;
            for (auto& s : ds) {
                const int nzp = (s.N + s.ptz - 1) / s.ptz, g = std::max(1, std::min({nzp, 8, d * nzp / s.N}));
                const double c = (double)s.N * g / nzp + 3.0 + 0.5 * g;
                all += c * tiles62(s.N) * ((nzp + g - 1) / g);
                longest = std::max(longest, c);
            }
            const double t = all / (512.0 * longest) < 1.0 ? longest : all / 512.0 + 0.5 * longest;
            if (d == 1 || t < best) best = t;
            if (d == dd) mine = t;
        }
        if (mine > best * (1 + 1e-12)) return 5;
    }
    std::printf("ok\n");
    return 0;
}
"""


VARIANTS = r"""
#include "ttsh_layout.h"
#include <cstdio>
using namespace ttsh;
int main()
{
    // the tiles that boxes are measured against, by number: a box holds the
    // tile and one cell around it
    const int tx[7] = {32, 16, 64, 16, 32, 32, 64}, ty[7] = {8, 16, 4, 8, 8, 16, 8};
    for (int N : {32, 33, 34, 36, 40, 64, 65, 66, 72, 128, 256}) {
        for (int v = -2; v < 9; ++v)
            if (rhs_fits(v, N) != (v >= 0 && v < 7 && N >= tx[v] + 2 && N >= ty[v] + 2)) return 1;
        for (int asked = -1; asked < 7; ++asked)
            for (int tuned = -1; tuned < 7; ++tuned)
                for (int engine = -1; engine < 7; ++engine) {
                    const RhsChoice c = choose_rhs(N, asked, tuned, engine);
                    const bool first = engine < 0;
                    if (asked >= 0 && !rhs_fits(first ? asked : engine, N)) {
                        if (c.engine != -1) return 2;  // refused
                        continue;
                    }
                    if (!rhs_fits(c.engine, N)) return 3;
                    if (asked < 0 && !rhs_fits(c.own, N)) return 4;
                    if (c.own != (asked >= 0 ? asked : rhs_fits(tuned, N) ? tuned : 1)) return 5;
                    if (c.engine != (first ? c.own : rhs_fits(engine, N) ? engine : 1)) return 6;
                }
    }
    std::printf("ok\n");
    return 0;
}
"""


@pytest.mark.parametrize("driver", [DRIVER, VARIANTS], ids=["depths", "variants"])
def test_layout(tmp_path, driver):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "driver.cpp").write_text(driver)
    exe = tmp_path / "driver"
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-I", CSRC,
                        str(tmp_path / "driver.cpp"), "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout + r.stderr)
