// CPU check of the MFMA scatter's tile maps (csrc/projector_maps.h: tile_row_off,
// row_atom, tile_vox), built with AddressSanitizer and UndefinedBehaviorSanitizer by
// tests/test_scatter_tiles_host.py.  The kernel dereferences their indices without
// bounds checks, so every one is checked against its definition, on random
// projector sets: wrapped and overlapping spheres, atoms without voxels, spheres
// wider than the cell (an atom that covers a point several times).
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "projector_maps.h"

using namespace qm;

static int fails = 0;
#define CHECK(c)                                                                                      \
    do {                                                                                              \
        if (!(c) && fails++ < 20) std::fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__); \
    } while (0)

static void run_case(std::mt19937 &rng, int nx, int ny, int nz, int natoms, int radius, int pile) {
    std::uniform_int_distribution<int> ux(0, nx - 1), uy(0, ny - 1), uz(0, nz - 1), um(1, 32), ur(0, radius);
    std::vector<int> nproj(natoms), proj_off(natoms + 1, 0), xyz;
    std::vector<int64_t> vox_off(natoms + 1, 0), tab_off(natoms + 1, 0);
    for (int a = 0; a < natoms; ++a) {
        nproj[a] = um(rng);
        const int r = ur(rng);
        const int cx = a < pile ? 1 : ux(rng), cy = a < pile ? 0 : uy(rng), cz = a < pile ? nz - 1 : uz(rng);
        int64_t V = 0;
        if (a % 5 != 4)
            for (int z = -r; z <= r; ++z)
                for (int y = -r; y <= r; ++y)
                    for (int x = -r; x <= r; ++x)
                        if (x * x + y * y + z * z <= r * r) {
                            xyz.insert(xyz.end(), {cx + x, cy + y, cz + z});
                            ++V;
                        }
        vox_off[a + 1] = vox_off[a] + V;
        tab_off[a + 1] = tab_off[a] + V * nproj[a];
        proj_off[a + 1] = proj_off[a] + nproj[a];
    }
    if (xyz.empty()) xyz.push_back(0);
    ProjectorMaps m;
    build_projector_maps(nx, ny, nz, natoms, nproj.data(), vox_off.data(), xyz.data(), nullptr, tab_off.data(),
                         proj_off.data(), 32, m, false);
    const int64_t vtot = vox_off[natoms];
    const int ncov = (int)m.cov_grid.size(), ntile = (ncov + kScatterTile - 1) / kScatterTile;
    CHECK((int)m.tile_row_off.size() == ntile + 1 && m.tile_row_off[0] == 0);
    CHECK(m.tile_row_off.back() == (int)m.row_atom.size());
    CHECK(m.tile_vox.size() == m.row_atom.size() * kScatterTile);
    std::vector<int> seen(vtot, 0);  // rows that hold the voxel
    for (int b = 0; b < ntile; ++b) {
        const int i0 = b * kScatterTile, r0 = m.tile_row_off[b], r1 = m.tile_row_off[b + 1];
        CHECK(r1 > r0);  // the kernel loads the first row unconditionally
        for (int r = r0; r < r1; ++r) {
            const int a = m.row_atom[r];
            CHECK(a >= 0 && a < natoms);
            bool any = false;
            for (int i = 0; i < kScatterTile; ++i) {
                const int v = m.tile_vox[(size_t)r * kScatterTile + 4 * (i & 15) + (i >> 4)];
                CHECK(v >= -1 && v < (int)vtot);
                if (v < 0) continue;
                any = true;
                CHECK(i0 + i < ncov);
                CHECK(m.atom[v] == a);
                if (i0 + i < ncov) CHECK(m.grid[v] == m.cov_grid[i0 + i]);
                ++seen[v];
            }
            CHECK(any);
        }
    }
    CHECK(std::all_of(seen.begin(), seen.end(), [](int n) { return n == 1; }));
}

int main() {
    std::mt19937 rng(20261001u);
    int cases = 0;
    for (int rep = 0; rep < 60; ++rep, ++cases) {
        const int natoms = 1 + rep % 13;
        run_case(rng, 5 + rep % 7, 4 + rep % 5, 4 + rep % 6, natoms, rep % 3 == 0 ? 6 : 3, rep % 4 == 0 ? natoms : 0);
    }
    run_case(rng, 24, 20, 18, 30, 5, 8);
    if (fails) {
        std::fprintf(stderr, "%d checks failed\n", fails);
        return 1;
    }
    std::printf("scatter tiles: %d cases ok\n", cases + 1);
    return 0;
}
