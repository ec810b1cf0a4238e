// Host model of the occupancy prefix of large levels: the tiles of bitmap words that hold any occupied
// cell get every word's prefix, the empty ones what emptyWordPrefixes stores, the rest stays a value that
// no prefix has. Every neighbourhood window of every occupied cell (rowRun, as the inter-cell and the
// weighted filter walk it) that holds any cell must start at that cell's rank, and every node must know its
// first rank. Prints the windows checked, and of them those that start in an empty tile.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "cell_order.h"

using namespace oc;

static const uint32_t UNWRITTEN = 0xDEADBEEFu;

struct Checked
{
    uint64_t windows = 0, acrossTiles = 0;
};

// cells: occupied bits of the level's bitmap (node * 32 * wordsPerNode + cell). Exits on a wrong rank.
static void check(uint32_t g, uint32_t nodes, uint64_t tile, const std::vector<uint64_t>& cells, Checked& sum)
{
    const uint64_t wordsPerNode = (rowsPerNode(g) * g + 31) / 32, words = nodes * wordsPerNode;
    std::vector<uint32_t> bits(words), rank(words + 1), prefix(words + 1, UNWRITTEN);
    for (uint64_t c : cells)
        bits[c >> 5] |= 1u << (c & 31);
    for (uint64_t w = 0; w < words; ++w)
        rank[w + 1] = rank[w] + static_cast<uint32_t>(__builtin_popcount(bits[w]));
    prefix[words] = rank[words];
    for (uint64_t base = 0; base < words; base += tile)
    {
        const uint64_t end = base + tile < words ? base + tile : words;
        if (rank[end] == rank[base])
            for (uint32_t thread = 0; thread < 4; ++thread)
                emptyWordPrefixes(base, end, wordsPerNode, thread, 4, [&](uint64_t w) { prefix[w] = rank[base]; });
        else
            for (uint64_t w = base; w < end; ++w)
                prefix[w] = rank[w];
    }
    auto fail = [&](const char* what, uint64_t at, uint32_t got, uint32_t want) {
        std::printf("g %u nodes %u tile %llu: %s %llu: %u, not %u\n", g, nodes, static_cast<unsigned long long>(tile),
                    what, static_cast<unsigned long long>(at), got, want);
        std::exit(1);
    };
    for (uint32_t k = 0; k <= nodes; ++k)
        if (prefix[k * wordsPerNode] != rank[k * wordsPerNode])
            fail("node", k, prefix[k * wordsPerNode], rank[k * wordsPerNode]);
    for (uint64_t c : cells)
    {
        const uint64_t node = c / (32 * wordsPerNode) * wordsPerNode;
        uint32_t x = 0, y = 0, z = 0;
        cellCoords(static_cast<uint32_t>(c - 32 * node), g, x, y, z);
        const uint32_t x0 = x > 0 ? x - 1 : 0, x1 = x + 1 < g ? x + 1 : x;
        const CellRows rows(y, z, g);
        for (int r = 0; r < 9; ++r)
        {
            if (!rows.has(r))
                continue;
            const uint32_t start = rows.start(r) + x0;
            const RowRun run     = rowRun(bits.data() + node, prefix.data() + node, start, x1 - x0 + 1);
            uint32_t count = 0, first = 0;
            for (uint32_t i = start; i <= rows.start(r) + x1; ++i)
            {
                const uint64_t w = node + (i >> 5);
                if ((bits[w] >> (i & 31)) & 1u)
                {
                    if (count++ == 0)
                        first = rank[w] + static_cast<uint32_t>(__builtin_popcount(bits[w] & ((1u << (i & 31)) - 1u)));
                }
            }
            if (run.count != count)
                fail("window's cells at cell", c, run.count, count);
            if (count && run.first != first)
                fail("window's first rank at cell", c, run.first, first);
            const uint64_t own = (node + (start >> 5)) / tile * tile;
            sum.windows += count != 0;
            sum.acrossTiles += count != 0 && rank[own + tile < words ? own + tile : words] == rank[own];
        }
    }
}

int main(int argc, char** argv)
{
    const uint64_t tile = argc > 1 ? std::strtoull(argv[1], nullptr, 10) : 2048;
    std::mt19937_64 rng(17);
    Checked sum;
    const uint32_t grids[] = {1, 2, 3, 5, 7, 12, 20, 31, 32, 33, 37, 48, 50, 64, 96, 99, 100, 104, 112, 128, 131, 160, 200, 250, 255};
    for (uint32_t g : grids)
    {
        const uint64_t perNode = 32 * ((rowsPerNode(g) * g + 31) / 32);
        for (uint32_t nodes : {1u, 2u, 5u})
        {
            // one cell at, before or after the first bit of every second tile, and clusters in between
            std::vector<uint64_t> cells;
            const uint64_t all = perNode * nodes;
            auto add = [&](uint64_t c) {
                // only cells of the grid: pencils at its upper faces hold rows outside it
                uint32_t x = 0, y = 0, z = 0;
                if (c >= all || c % perNode >= rowsPerNode(g) * g)
                    return;
                cellCoords(static_cast<uint32_t>(c % perNode), g, x, y, z);
                if (y < g && z < g)
                    cells.push_back(c);
            };
            for (uint64_t at = 32 * tile; at < all; at += 64 * tile)
            {
                const uint64_t shift = rng() % 3;  // 0 to 2 cells past the tile's first bit
                add(at + shift);
                if (rng() % 2)
                    add(at + shift + 1 + rng() % 40);
            }
            check(g, nodes, tile, cells, sum);
            for (int k = 0; k < 20; ++k)
            {
                const uint64_t c = rng() % all;
                for (int j = 0; j < 8; ++j)
                    add(c + rng() % (2ull * g + 2));
            }
            check(g, nodes, tile, cells, sum);
        }
    }
    std::printf("windows %llu, starting in an empty tile %llu\n", static_cast<unsigned long long>(sum.windows),
                static_cast<unsigned long long>(sum.acrossTiles));
    return 0;
}
