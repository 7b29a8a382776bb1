"""Whether TMS_BC's outflow and inflow lists lie apart (sweep_lists.h).

Against a look at every cell within the limit, on small random grids with
distances around it, and, for two faces of 256 x 256 cells that lie just apart,
in less than half the time of that look (1331 cells for each inflow cell)."""
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "lattice-boltzmann-method_amd")

SRC = r"""
#include <chrono>
#include <cstdio>
#include <random>
#include "sweep_lists.h"
static bool by_marks(const std::vector<int>& a, const std::vector<int>& b, int nx, int ny, int nz, int far)
{
    std::vector<uint8_t> near((size_t)nx * ny * nz, 0);
    bool apart = true;
    for (int t : a) near[t] = 1;
    for (int t : b) {
        const int i = t / (ny * nz), j = t / nz % ny, k = t % nz;
        for (int x = std::max(i - far, 0); x <= std::min(i + far, nx - 1); ++x)
            for (int y = std::max(j - far, 0); y <= std::min(j + far, ny - 1); ++y)
                for (int z = std::max(k - far, 0); z <= std::min(k + far, nz - 1); ++z)
                    if (near[((int64_t)x * ny + y) * nz + z]) apart = false;
        if (!apart) break;
    }
    return apart;
}
static double seconds()
{
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}
int main()
{
    std::mt19937 g(11);
    int bad = 0, yes = 0, n = 0;
    for (int r = 0; r < 20000; ++r) {
        const int nx = 1 + g() % 24, ny = 1 + g() % 24, nz = 1 + g() % 24, far = g() % 7, cells = nx * ny * nz;
        std::vector<int> a(g() % 4), b(g() % 4);
        for (int& c : a) c = g() % cells;
        for (int& c : b) c = g() % cells;
        const bool want = by_marks(a, b, nx, ny, nz, far);
        yes += want;
        ++n;
        bad += lbm::sweeps_apart(a, b, ny, nz, far) != want;
    }
    std::vector<int> a, b;
    const int m = 258;
    for (int j = 1; j < m - 1; ++j)
        for (int k = 1; k < m - 1; ++k) {
            a.push_back((1 * m + j) * m + k);
            b.push_back((7 * m + j) * m + k);
        }
    a.push_back((13 * m + 5) * m + 5);
    double t0 = seconds();
    const bool w = by_marks(a, b, 16, m, m, 5);
    const double slow = seconds() - t0;
    t0 = seconds();
    const bool q = lbm::sweeps_apart(a, b, m, m, 5);
    const double fast = seconds() - t0;
    printf("%d of %d wrong (%d apart); faces %d %d, %.4f and %.4f s\n", bad, n, yes, w, q, slow, fast);
    return bad || yes < n / 20 || yes > n - n / 20 || !w || !q || fast > slow / 2;
}
"""


def test_lists_apart(tmp_path):
    src, exe = tmp_path / "s.cpp", tmp_path / "s"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{PKG}/csrc", "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    print(r.stdout)
