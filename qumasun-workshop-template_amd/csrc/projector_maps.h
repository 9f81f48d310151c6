// Host-side index maps of a projector set: the part of qm_set_projectors that
// needs no device, kept free of HIP so that it also builds with a plain C++
// compiler (the CPU tests build it with AddressSanitizer).
//
// Inputs follow qm_set_projectors (include/qumasun_hip.h): atom a owns voxels
// vox_off[a] .. vox_off[a+1]-1 with unwrapped coordinates vox_xyz[3 v ..],
// nproj[a] projectors whose table is table[tab_off[a] + w V_a + v] (V_a voxels,
// projector-major, as the reference's SvF tables, PseudoPotNonlocal_SvF2_kpoint.h
// :911-1178), and projector ids proj_off[a] .. proj_off[a+1]-1.
#pragma once

#include <algorithm>
#include <cstdint>
#include <numeric>
#include <vector>

namespace qm {

constexpr int kProjChunk = 512;     // voxels per projection work item (4 waves x 128)
constexpr int kScatterBlock = 256;  // covered points per scatter workgroup
constexpr int kScatterSlots = 8;    // atoms whose coefficients a scatter workgroup stages in LDS
constexpr int kScatterTile = 64;    // covered points per tile of the MFMA scatter (4 x 16)

// periodic wrap of a grid coordinate into 0 .. n-1
inline int wrap_index(int i, int n) {
    const int r = i % n;
    return r < 0 ? r + n : r;
}

struct ProjectorMaps {
    std::vector<int> grid, atom;  // [vtot] wrapped grid index and owner atom of every voxel
    // owner-computes scatter: covered grid points in increasing order, each with
    // its voxels cov_vox[cov_off[i] .. cov_off[i+1]-1]
    std::vector<int> cov_grid, cov_off, cov_vox;
    std::vector<int> atom_order;  // heaviest atoms (V_a M_a) first
    // voxel-major tables padded to mpad projectors: tabp[v mpad + w] (with_tables)
    std::vector<double> tabp64;
    std::vector<float> tabp32;
    // projection work items (chunks of kProjChunk voxels of one atom), the
    // atoms' ranges of them, each projector's atom, the launch order
    std::vector<int> chunk_atom, chunk_v0, atom_chunk_off, proj_atom, item_order;
    // per scatter block of kScatterBlock covered points: its distinct atoms
    // (at most kScatterSlots staged) and each voxel entry's slot (-1: not staged)
    std::vector<int> block_atom_off, block_atoms, cov_slot;
    // per tile of kScatterTile covered points, one row per atom that covers any
    // of them: the atom's voxel at the tile's point 16 t + j is
    // tile_vox[64 row + 4 j + t], -1 where its sphere does not reach.  An atom
    // that covers a point more than once (a sphere wider than the cell) has
    // further rows, so that every entry is in exactly one.
    std::vector<int> tile_row_off, row_atom, tile_vox;
};

inline void build_projector_maps(int nx, int ny, int nz, int natoms, const int *nproj, const int64_t *vox_off,
                                 const int *vox_xyz, const double *table, const int64_t *tab_off,
                                 const int *proj_off, int mpad, ProjectorMaps &m, bool with_tables = true) {
    const int64_t vtot = vox_off[natoms];
    const int ptot = proj_off[natoms];
    m.grid.assign(vtot, 0);
    m.atom.assign(vtot, 0);
    for (int a = 0; a < natoms; ++a)
        for (int64_t v = vox_off[a]; v < vox_off[a + 1]; ++v) {
            m.grid[v] = wrap_index(vox_xyz[3 * v], nx) +
                        nx * (wrap_index(vox_xyz[3 * v + 1], ny) + ny * wrap_index(vox_xyz[3 * v + 2], nz));
            m.atom[v] = a;
        }
    // covered-point map: voxels sorted by grid point, in their own order at each
    // (a counting sort over the grid)
    std::vector<int> at((size_t)nx * ny * nz + 1, 0);
    for (int64_t v = 0; v < vtot; ++v) ++at[m.grid[v] + 1];
    m.cov_grid.clear();
    m.cov_off.clear();
    for (size_t g = 0; g + 1 < at.size(); ++g) {
        if (at[g + 1] > 0) {
            m.cov_grid.push_back((int)g);
            m.cov_off.push_back(at[g]);
        }
        at[g + 1] += at[g];
    }
    m.cov_vox.resize(vtot);
    for (int64_t v = 0; v < vtot; ++v) m.cov_vox[at[m.grid[v]]++] = (int)v;
    m.cov_off.push_back((int)vtot);
    const int ncov = (int)m.cov_grid.size();
    m.atom_order.resize(natoms);
    std::iota(m.atom_order.begin(), m.atom_order.end(), 0);
    std::stable_sort(m.atom_order.begin(), m.atom_order.end(), [&](int x, int y) {
        return (vox_off[x + 1] - vox_off[x]) * nproj[x] > (vox_off[y + 1] - vox_off[y]) * nproj[y];
    });
    // padded voxel-major tables and the projection work list
    m.tabp64.assign(with_tables ? (size_t)vtot * mpad : 0, 0.0);
    m.tabp32.assign(with_tables ? (size_t)vtot * mpad : 0, 0.0f);
    m.chunk_atom.clear();
    m.chunk_v0.clear();
    m.atom_chunk_off.assign(natoms + 1, 0);
    m.proj_atom.assign(ptot, 0);
    for (int a = 0; a < natoms; ++a) {
        const int64_t V = vox_off[a + 1] - vox_off[a];
        for (int w = 0; w < nproj[a]; ++w) {
            m.proj_atom[proj_off[a] + w] = a;
            for (int64_t v = 0; with_tables && v < V; ++v) {
                const double val = table[tab_off[a] + w * V + v];
                m.tabp64[(size_t)(vox_off[a] + v) * mpad + w] = val;
                m.tabp32[(size_t)(vox_off[a] + v) * mpad + w] = (float)val;
            }
        }
        for (int64_t v0 = 0; v0 < V; v0 += kProjChunk) {
            m.chunk_atom.push_back(a);
            m.chunk_v0.push_back((int)v0);
        }
        m.atom_chunk_off[a + 1] = (int)m.chunk_atom.size();
    }
    // launch order of the work items: by the (wrapped) z, then y, of each
    // chunk's first voxel, so that the chunks of neighbouring atoms that read
    // the same grid lines run together on one XCD and share its L2
    const int nchunk = (int)m.chunk_atom.size();
    std::vector<int64_t> key(nchunk);
    for (int it = 0; it < nchunk; ++it) {
        const int64_t v = vox_off[m.chunk_atom[it]] + m.chunk_v0[it];
        key[it] = (int64_t)wrap_index(vox_xyz[3 * v + 2], nz) * ny + wrap_index(vox_xyz[3 * v + 1], ny);
    }
    m.item_order.resize(nchunk);
    std::iota(m.item_order.begin(), m.item_order.end(), 0);
    std::stable_sort(m.item_order.begin(), m.item_order.end(), [&](int a, int b) { return key[a] < key[b]; });
    // scatter blocks: distinct atoms of their entries, and every entry's slot
    const int nb = (ncov + kScatterBlock - 1) / kScatterBlock;
    m.block_atom_off.assign(nb + 1, 0);
    m.block_atoms.clear();
    m.cov_slot.assign(vtot, -1);
    for (int b = 0; b < nb; ++b) {
        std::vector<int> list;
        const int i0 = b * kScatterBlock, i1 = std::min(ncov, i0 + kScatterBlock);
        for (int i = i0; i < i1; ++i)
            for (int e = m.cov_off[i]; e < m.cov_off[i + 1]; ++e) {
                const int a = m.atom[m.cov_vox[e]];
                int s = -1;
                for (int q = 0; q < (int)list.size(); ++q)
                    if (list[q] == a) s = q;
                if (s < 0 && (int)list.size() < kScatterSlots) {
                    list.push_back(a);
                    s = (int)list.size() - 1;
                }
                m.cov_slot[e] = s;
            }
        m.block_atoms.insert(m.block_atoms.end(), list.begin(), list.end());
        m.block_atom_off[b + 1] = (int)m.block_atoms.size();
    }
    if (m.block_atoms.empty()) m.block_atoms.push_back(0);
    // MFMA scatter: every entry goes to the first row of its atom, in this tile,
    // that has no entry yet at its point
    const int ntile = (ncov + kScatterTile - 1) / kScatterTile;
    m.tile_row_off.assign(ntile + 1, 0);
    m.row_atom.clear();
    m.tile_vox.clear();
    for (int b = 0; b < ntile; ++b) {
        const int i0 = b * kScatterTile, i1 = std::min(ncov, i0 + kScatterTile);
        const size_t r0 = m.row_atom.size();
        for (int i = i0; i < i1; ++i) {
            const int p = 4 * ((i - i0) & 15) + ((i - i0) >> 4);
            for (int e = m.cov_off[i]; e < m.cov_off[i + 1]; ++e) {
                const int a = m.atom[m.cov_vox[e]];
                size_t r = r0;
                while (r < m.row_atom.size() &&
                       (m.row_atom[r] != a || m.tile_vox[r * kScatterTile + p] >= 0))
                    ++r;
                if (r == m.row_atom.size()) {
                    m.row_atom.push_back(a);
                    m.tile_vox.resize((r + 1) * kScatterTile, -1);
                }
                m.tile_vox[r * kScatterTile + p] = m.cov_vox[e];
            }
        }
        m.tile_row_off[b + 1] = (int)m.row_atom.size();
    }
}

}  // namespace qm
