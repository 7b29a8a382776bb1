// Host side of TMS_BC's interface-cell lists.
#pragma once
#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <map>
#include <vector>

namespace lbm {

// Cells (i ny + j) nz + k of a grid in blocks of `step` cells, with the bounds of
// each block's cells.
struct CellBlocks {
    struct Cell {
        int x[3];
    };
    struct Block {
        Cell lo, hi;
        std::vector<Cell> cells;
    };
    std::map<int64_t, Block> blocks;  // key: block indices, 21 bits each
    static int64_t key(int i, int j, int k) { return ((int64_t)i << 42) | ((int64_t)j << 21) | k; }
    CellBlocks(const std::vector<int>& list, int ny, int nz, int step)
    {
        Block* last = nullptr;
        int64_t last_key = -1;
        for (int c : list) {
            const Cell p{{c / (ny * nz), c / nz % ny, c % nz}};
            const int64_t at = key(p.x[0] / step, p.x[1] / step, p.x[2] / step);
            if (at != last_key) {  // (lists run along the cells: mostly the same block again)
                const auto r = blocks.try_emplace(at);
                last = &r.first->second;
                last_key = at;
                if (r.second) last->lo = last->hi = p;
            }
            for (int d = 0; d < 3; ++d) {
                last->lo.x[d] = std::min(last->lo.x[d], p.x[d]);
                last->hi.x[d] = std::max(last->hi.x[d], p.x[d]);
            }
            last->cells.push_back(p);
        }
    }
};

// Whether every cell of `a` lies more than `far` cells from every cell of `b` in some
// direction.  Both lists are sorted into blocks of far + 1 cells; a block's
// bounds are held against those of the 27 blocks around it in the other list, and
// the cells themselves only where the bounds come near.  (A look at the
// (2 far + 1)^3 cells around each cell of `b` took 0.11 s for two faces of 256 x 256
// cells six apart, this 0.018.)
inline bool sweeps_apart(const std::vector<int>& a, const std::vector<int>& b, int ny, int nz, int far)
{
    if (a.empty() || b.empty()) return true;
    const CellBlocks A(a, ny, nz, far + 1), B(b, ny, nz, far + 1);
    using Cell = CellBlocks::Cell;
    auto apart = [&](const Cell& lo, const Cell& hi, const Cell& lo2, const Cell& hi2) {
        for (int d = 0; d < 3; ++d)
            if (lo2.x[d] - hi.x[d] > far || lo.x[d] - hi2.x[d] > far) return true;
        return false;
    };
    for (const auto& kb : B.blocks)
        for (int i = -1; i <= 1; ++i)
            for (int j = -1; j <= 1; ++j)
                for (int k = -1; k <= 1; ++k) {
                    const int64_t at = kb.first + i * ((int64_t)1 << 42) + j * (1 << 21) + k;
                    const auto ka = A.blocks.find(at);
                    if (ka == A.blocks.end()) continue;
                    const auto &x = ka->second, &y = kb.second;
                    if (apart(x.lo, x.hi, y.lo, y.hi)) continue;
                    for (const Cell& q : y.cells)
                        for (const Cell& p : x.cells)
                            if (!apart(p, p, q, q)) return false;
                }
    return true;
}

}  // namespace lbm
