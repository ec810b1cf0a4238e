// Order of the cells of a node's subsampling grid, and the rank dictionary over them (occupancy bitmap
// and popcount prefix of its words): plain arithmetic for the kernels and for host code.
#pragma once

#include <cstdint>

namespace oc {

// Cell index of a node grid. The x-rows (fixed y, z) are grouped into 4 x 4 pencils, pencils in
// (z / 4, y / 4) order and rows inside a pencil in (z % 4, y % 4) order; a cell is row * g + x.
// A row stays one contiguous run of bits (and of dense ranks), and the 9 rows a cell's 3x3x3
// neighbourhood touches lie a few rows apart instead of a whole z-plane apart.
constexpr uint32_t PENCIL = 4;

constexpr uint32_t pencilsPerAxis(uint32_t g)
{
    return (g + PENCIL - 1) / PENCIL;
}

constexpr uint64_t rowsPerNode(uint32_t g)
{
    const uint64_t p = pencilsPerAxis(g);
    return p * p * PENCIL * PENCIL;
}

constexpr uint32_t rowIndex(uint32_t y, uint32_t z, uint32_t g)
{
    const uint32_t p = pencilsPerAxis(g);
    return (((z / PENCIL) * p + (y / PENCIL)) * PENCIL + (z % PENCIL)) * PENCIL + (y % PENCIL);
}

constexpr void rowCoords(uint32_t row, uint32_t g, uint32_t& y, uint32_t& z)
{
    const uint32_t p = pencilsPerAxis(g), pencil = row / (PENCIL * PENCIL), inside = row % (PENCIL * PENCIL);
    y = (pencil % p) * PENCIL + inside % PENCIL;
    z = (pencil / p) * PENCIL + inside / PENCIL;
}

// A cell's coordinates from its index, g the same for all cells of a build: shifts where it is a power of
// two, integer divisions (some 25 instructions each) where not.
constexpr void cellCoords(uint32_t cell, uint32_t g, uint32_t& x, uint32_t& y, uint32_t& z)
{
    if (g >= PENCIL && (g & (g - 1)) == 0)
    {
        const uint32_t s = static_cast<uint32_t>(__builtin_ctz(g)), p = g / PENCIL;
        const uint32_t row = cell >> s, pencil = row / (PENCIL * PENCIL), inside = row % (PENCIL * PENCIL);
        x = cell & (g - 1);
        y = (pencil & (p - 1)) * PENCIL + inside % PENCIL;
        z = (pencil >> __builtin_ctz(p)) * PENCIL + inside / PENCIL;
        return;
    }
    x = cell % g;
    rowCoords(cell / g, g, y, z);
}

// The 3 x 3 x-rows around a cell: rowIndex is a sum of a part in y and one in z, so the first cells of
// the nine rows are nine sums.
struct CellRows
{
    uint32_t y[3] = {}, z[3] = {};    // the parts, in cells
    bool inY[3] = {}, inZ[3] = {};    // in the grid
    constexpr CellRows(uint32_t cy, uint32_t cz, uint32_t g)
    {
        const uint32_t p = pencilsPerAxis(g);
        for (uint32_t k = 0; k < 3; ++k)
        {
            const uint32_t ny = cy + k - 1, nz = cz + k - 1;  // below zero: above any g
            inY[k] = ny < g;
            inZ[k] = nz < g;
            y[k]   = (ny / PENCIL * (PENCIL * PENCIL) + ny % PENCIL) * g;
            z[k]   = (nz / PENCIL * p * (PENCIL * PENCIL) + nz % PENCIL * PENCIL) * g;
        }
    }
    constexpr bool has(int r) const { return inY[r / 3] && inZ[r % 3]; }
    constexpr uint32_t start(int r) const { return y[r / 3] + z[r % 3]; }
};

// The occupied cells among `span` <= 3 consecutive cells of a node, from cell `start` on: how many, and
// the dense index of the first (meaningless if there is none). The cells lie in one word or two; the
// index comes from the prefix of the first of them, also where only the second holds any.
struct RowRun
{
    uint32_t first, count;
};

constexpr RowRun rowRun(const uint32_t* bits, const uint32_t* prefix, uint32_t start, uint32_t span)
{
    const uint32_t w = start >> 5, b = start & 31;
    uint64_t v       = bits[w];
    if (b + span > 32)
        v |= static_cast<uint64_t>(bits[w + 1]) << 32;
    const uint32_t in = static_cast<uint32_t>(v >> b) & ((1u << span) - 1u);
    return RowRun{prefix[w] + static_cast<uint32_t>(__builtin_popcount(static_cast<uint32_t>(v) & ((1u << b) - 1u))),
                  static_cast<uint32_t>(__builtin_popcount(in))};
}

// store(w) for the words w of [base, end), a stretch of the bitmap without any occupied cell, whose
// prefixes are read all the same: the first word of every node (where its cells start) and the stretch's
// last word, in which a row's window may begin whose cells lie in the word after it (rowRun; a stretch
// ends inside a row where rows do not divide it, as with g = 96 or 100). Thread `thread` of `threads`
// does its part.
template <typename Store>
constexpr void emptyWordPrefixes(uint64_t base, uint64_t end, uint64_t wordsPerNode, uint32_t thread, uint32_t threads,
                                 Store store)
{
    for (uint64_t w = ((base + wordsPerNode - 1) / wordsPerNode + thread) * wordsPerNode; w < end;
         w += threads * wordsPerNode)
        store(w);
    if (thread == 0)
        store(end - 1);
}

}  // namespace oc
