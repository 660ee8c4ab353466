// Rules of the launch plans (rg_plan.h), checked on the host: exit code 0 if
// all hold, otherwise the failing rule is printed.
#include <cstdio>

#include "rg_plan.h"

static int bad = 0;
#define EXPECT(cond, ...)                \
    do {                                 \
        if (!(cond)) {                   \
            std::printf(__VA_ARGS__);    \
            std::printf(": %s\n", #cond); \
            ++bad;                       \
        }                                \
    } while (0)

// values of symmetric 3 x 3 blocks: 14 stored slots of 9 entries
static bool marches(int e0, int e1, int e2, int vsize, int cu = 256)
{
    const rg::MarchArgs m = rg::march_args(e0 + 1, e1 + 1, e2 + 1, cu);
    const int64_t ld = ((int64_t)(e0 + 1) * (e1 + 1) * (e2 + 1) + 63) / 64 * 64;
    return rg::march_applies(m, 14 * 9 * ld * vsize, vsize, cu);
}

// the reducing kernels write one partial per workgroup: no plan has more of
// them than partials (kMaxGrid)
static void march_fits_the_partials()
{
    const int wide[][3] = {{7600, 7600, 1}, {1850, 1850, 20}, {2400, 1600, 3}, {60, 90000, 2}, {90000, 60, 2}, {3000, 3000, 4}};
    for (auto& e : wide)
        for (int vsize : {4, 8}) {
            const rg::MarchArgs m = rg::march_args(e[0] + 1, e[1] + 1, e[2] + 1, 256);
            EXPECT(!marches(e[0], e[1], e[2], vsize) || rg::march_grid(m) <= rg::kMaxGrid, "%d x %d x %d", e[0], e[1], e[2]);
        }
    EXPECT(!marches(7600, 7600, 1, 8), "137,922 workgroups");
    EXPECT(marches(96, 96, 96, 8) && marches(96, 96, 96, 4) && marches(1400, 1300, 1, 8), "grids that march");
}

// every node belongs to one tile and segment, and a tile fits the workgroup
static void march_covers()
{
    for (int n0 : {2, 3, 9, 65, 97, 170, 171, 700})
        for (int n1 : {2, 14, 97, 513})
            for (int n2 : {2, 5, 97, 9001}) {
                const rg::MarchArgs m = rg::march_args(n0, n1, n2, 256);
                EXPECT((m.tx + 2) * (m.ty + 2) <= rg::kMarchThreads, "%d x %d x %d", n0, n1, n2);
                EXPECT((int64_t)m.tx * m.gx >= n0 && m.tx * (m.gx - 1) < n0, "%d x %d x %d", n0, n1, n2);
                EXPECT((int64_t)m.ty * m.gy >= n1 && m.ty * (m.gy - 1) < n1, "%d x %d x %d", n0, n1, n2);
            }
}

// grids whose tiles leave most threads without a node, or most CUs without a
// tile, gather (measured slower marching); the ones beside them march
static void march_fills_the_chip()
{
    EXPECT(!marches(2, 2, 60000, 8) && !marches(2, 2, 60000, 4), "3 x 3 nodes per plane");
    EXPECT(!marches(8, 8, 9000, 8) && !marches(8, 8, 9000, 4), "9 x 9 nodes per plane");
    EXPECT(!marches(10, 10, 7000, 8) && !marches(11, 11, 5000, 8) && marches(12, 12, 4000, 8), "121, 144 and 169 nodes per plane");
    EXPECT(!marches(64, 63, 66, 8) && marches(64, 64, 64, 8), "140 and 195 workgroups of 5 planes");
    EXPECT(!marches(228, 228, 30, 4) && marches(228, 228, 30, 8), "130 workgroups");
    EXPECT(!marches(30, 30, 900, 4) && marches(30, 30, 900, 8), "tiles of 8 x 31 nodes");
    EXPECT(marches(200, 180, 40, 4) && marches(24, 24, 1500, 4) && marches(1000, 900, 3, 4), "filled tiles");
}

// assembly tiles fit a workgroup's threads and LDS and cover the grid; short
// lines are whole, the closed form keeps the wide tile otherwise
static void assembly_tiles()
{
    const int64_t sides[] = {2, 3, 4, 5, 8, 9, 17, 31, 32, 33, 49, 64, 65, 66, 71, 97, 129, 1000};
    for (int dim : {2, 3})
        for (int nb : {1, 2, 3, 4}) {
            const int npw = 64 / (nb * nb);
            for (int64_t n0 : sides)
                for (int64_t n1 : sides)
                    for (int64_t n2 : {2, 7, 300})
                        for (bool staged : {false, true}) {
                            const int64_t nn[3] = {n0, n1, n2};
                            const rg::AsmTile t = rg::asm_tile(dim, nn, npw, staged);
                            const int around = (t.wx + 1) * (t.wy + 1) * (dim == 3 ? t.wz + 1 : 1);
                            EXPECT(t.wx * t.wy * t.wz <= 4 * npw && around <= rg::asm_tile_elements(dim, npw) &&
                                       t.wx * t.gx >= n0 && t.wy * t.gy >= n1 && (dim == 2 ? t.gz == 1 : t.wz * t.gz >= n2),
                                   "%d-D %d equations %lld x %lld x %lld", dim, nb, (long long)n0, (long long)n1, (long long)n2);
                            EXPECT(rg::asm_is_wide(t, dim, npw) || staged || t.wx == n0, "%lld", (long long)n0);
                        }
        }
    const int64_t thin[3] = {4, 4, 4001}, cube[3] = {97, 97, 97}, over[3] = {65, 65, 41};
    EXPECT(rg::asm_tile(3, thin, 64, false).wx == 4 && rg::asm_tile(3, thin, 64, true).wx == 4, "short lines");
    EXPECT(rg::asm_is_wide(rg::asm_tile(3, cube, 7, true), 3, 7), "97 nodes, 3 equations");
    EXPECT(!rg::asm_is_wide(rg::asm_tile(3, over, 64, true), 3, 64) && rg::asm_is_wide(rg::asm_tile(3, over, 64, false), 3, 64),
           "65 nodes");
}

// a batch's schedule: every tile of every system once, a workgroup has at most
// one tile of a system, and all lists are subsequences of one order of the
// systems -- run in that order every system finds all its workgroups
static void schedules_end()
{
    unsigned seed = 1;
    auto rnd = [&](int n) { return (int)((seed = seed * 1664525u + 1013904223u) >> 8) % n; };
    for (int round = 0; round < 300; ++round) {
        const int blocks = 1 + rnd(256), systems = 1 + rnd(60);
        std::vector<double> time;
        std::vector<int> tiles, first;
        std::vector<int32_t> system, rank;
        for (int j = 0; j < systems; ++j) {
            tiles.push_back(1 + rnd(rnd(3) ? std::min(blocks, 9) : blocks));
            time.push_back(1 + rnd(rnd(2) ? 3 : 1000));
        }
        rg::resident_schedule(time, tiles, blocks, first, system, rank);
        int total = 0;
        for (int t : tiles) total += t;
        EXPECT((int)system.size() == total && (int)first.size() == blocks + 1 && first.back() == total, "round %d", round);
        std::vector<std::vector<char>> seen(systems);
        for (int j = 0; j < systems; ++j) seen[j].assign(tiles[j], 0);
        for (size_t k = 0; k < system.size(); ++k) EXPECT(!seen[system[k]][rank[k]]++, "round %d", round);
        // workgroups advance past a system once all its tiles are at its head
        std::vector<int> at(first.begin(), first.end() - 1);
        int left = total;
        for (bool moved = true; moved && left;) {
            moved = false;
            std::vector<int> heads(systems, 0);
            for (int b = 0; b < blocks; ++b)
                if (at[b] < first[b + 1]) ++heads[system[at[b]]];
            for (int b = 0; b < blocks; ++b)
                if (at[b] < first[b + 1] && heads[system[at[b]]] == tiles[system[at[b]]]) {
                    ++at[b];
                    --left;
                    moved = true;
                }
        }
        EXPECT(left == 0, "round %d: %d blocks, %d systems stuck", round, blocks, systems);
    }
}

// one-launch tiles hold every node, within the rows and cells of a workgroup
static void one_launch_tiles()
{
    const int64_t grids[][3] = {{2, 2, 1}, {3, 2501, 1}, {701, 701, 1}, {71, 70, 68}, {4, 4, 2001}, {2, 301, 301}, {65, 65, 65}};
    for (auto& n : grids) {
        const int dim = n[2] == 1 ? 2 : 3, rows = 512 * (dim == 2 ? 4 : 3), cells = rows + 3 * 512;
        int t[3] = {1, 1, 1};
        if (!rg::resident_tiles(dim, n, rows, cells, 256, t, 0.0)) continue;
        if (dim == 2) t[2] = 1;
        int64_t tiles = 1, vol = 1, pad = 1;
        for (int d = 0; d < dim; ++d) {
            tiles *= (n[d] + t[d] - 1) / t[d];
            vol *= t[d];
            pad *= t[d] + 2;
        }
        EXPECT(tiles <= 256 && vol <= rows && pad <= cells, "%lld x %lld x %lld", (long long)n[0], (long long)n[1], (long long)n[2]);
    }
}

int main()
{
    schedules_end();
    one_launch_tiles();
    assembly_tiles();
    march_fills_the_chip();
    march_fits_the_partials();
    march_covers();
    return bad != 0;
}
