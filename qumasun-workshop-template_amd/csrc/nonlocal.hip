// Nonlocal Kleinman-Bylander apply and its position derivative for gfx950.
//
//   Hpsi += sum_a e^{-ik.r} P_a diag(E_a dV) P_a^T e^{+ik.r} psi
//
// Mathematics: ProjectionPP_bundle_1 / _2 (PseudoPotNonlocal_SvF2_kpoint.h:3910-4236)
// with mInnerNonlocalPsi_v4/_v6_bundle (4463-4758), the Bloch phases of
// mCreateBlochExp (3537-3618) and the force sums of ForceNonlocal_bundle
// (3629-3731, inner products of mInnerNonlocalPsi_diff_bundle 4775-4880).
//
// GPU structure (replaces per-atom DGEMM_t / DGEMM_n calls, host Bloch loops,
// host-side MPI reductions and one AddSubgrid launch per atom colour):
//   1. project: one launch over (voxel chunk, 16-column band tile) work items
//      of every atom, so spheres of any size balance by construction.  Each
//      wave gathers 256 voxels x 16 SoA columns straight from the grid, applies
//      e^{+ik.r}, and multiplies by the voxel-major projector table on MFMA
//      (16 projectors x 16 columns, K = voxels); the four waves of a chunk and
//      then the chunks of an atom are summed in FP64 in a fixed order, and
//      E_w dV is folded in (coef).
//   2. scatter: owner-computes over the grid points covered by any sphere.
//      Each covered point sums the contributions of all atoms whose sphere
//      contains it for a tile of columns, so overlapping spheres need no
//      atomics or colouring, tables are read once per tile, and the result is
//      deterministic.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "qm_internal.h"
#include "qm_mfma.h"

namespace qm {
namespace {

// Workgroup numbering: hardware block b runs on XCD b % 8, so giving each XCD a
// contiguous range of logical blocks puts consecutive logical blocks (the
// column groups of one item or point block) on one XCD, where they share its
// L2 for the projector table rows and entry lists.  Returns -1 past the end.
__device__ __forceinline__ int xcd_block(int nblk, int per_xcd) {
    const int b = blockIdx.x;
    const int lb = (b & 7) * per_xcd + (b >> 3);
    return lb < nblk ? lb : -1;
}

template <typename T>
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// part[(item * 16 MT + w) * ncol + col] = <p_w | e^{ik.r} psi>_col summed over the
// item's voxels (col = real SoA column n * NC + c), for the GT 16-column tiles
// of column group g (logical block = item * groups + g) and the MT 16-row
// projector tiles of the table (rows padded to 16 MT).  Each wave takes kProjChunk / 4 voxels in
// sub-chunks of 64.  Per sub-chunk it reads its block of the voxel-major
// projector table once, as the MFMA A operand of all GT tiles; per tile the
// 64 x 16 block of (phase-rotated) psi values is gathered with lanes along
// voxels (coalesced along x runs) into the wave's own LDS stage and fed to
// MFMA as the B operand.  The stage is private to the wave, so no workgroup
// barrier is needed until the final reduction over the four waves.
constexpr int PJ_VPW = kProjChunk / 4;  // voxels per wave
constexpr int PJ_SUB = 64;              // voxels per LDS sub-chunk
template <typename T, int NC, bool PH, int GT, int MT>
__global__ __launch_bounds__(256) void nl_project_kernel(double *__restrict__ part, const T *__restrict__ psi,
                                                         int64_t ng, int ncol, const int *__restrict__ chunk_atom,
                                                         const int *__restrict__ chunk_v0,
                                                         const int64_t *__restrict__ vox_off,
                                                         const int *__restrict__ vox_grid, const T *__restrict__ tabp,
                                                         const T *__restrict__ phase,
                                                         const int *__restrict__ item_order, int groups, int nblk,
                                                         int per_xcd) {
    constexpr int MPAD = 16 * MT;
    using M = Mfma<T>;
    using acc_t = typename M::acc_t;
    __shared__ T stage[4][PJ_SUB][16 + 1];
    __shared__ double red[4][16 * 16];
    const int lb = xcd_block(nblk, per_xcd);
    if (lb < 0) return;  // the whole workgroup
    const int slot = lb / groups;
    const int item = item_order[slot];
    const int c0 = (lb - slot * groups) * 16 * GT;
    const int a = chunk_atom[item];
    const int64_t vg0 = vox_off[a];
    const int V = (int)(vox_off[a + 1] - vg0);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int j = lane & 15, g = lane >> 4;
    const int vb = chunk_v0[item] + wave * PJ_VPW;
    acc_t acc[GT][MT];
#pragma unroll
    for (int t = 0; t < GT; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = acc_t{0, 0, 0, 0};
    for (int sc = 0; sc < PJ_VPW / PJ_SUB; ++sc) {
        const int vs = vb + sc * PJ_SUB;
        if (vs >= V) break;  // wave-uniform: the rest of the wave's voxels are past the sphere
        // A[w = 16 mt + j][k = g] of the 16 k-steps of this sub-chunk
        T av[MT][PJ_SUB / 4];
#pragma unroll
        for (int s = 0; s < PJ_SUB / 4; ++s) {
            const int v = vs + 4 * s + g;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) av[mt][s] = v < V ? tabp[(vg0 + v) * MPAD + 16 * mt + j] : T(0);
        }
        // the lane's voxel for the gathers
        const int v = vs + lane;
        const bool in = v < V;
        const int64_t vid = vg0 + (in ? v : 0);
        const int gi = in ? vox_grid[vid] : 0;
        T cs = T(1), sn = T(0);
        if constexpr (PH) {
            cs = phase[2 * vid];
            sn = phase[2 * vid + 1];
        }
        // all GT x 16 gathers first, so that they are in flight together
        T gv[GT][16];
#pragma unroll
        for (int t = 0; t < GT; ++t)
#pragma unroll
            for (int jj = 0; jj < 16; ++jj) {
                const int col = c0 + 16 * t + jj;
                gv[t][jj] = (in && col < ncol) ? psi[(int64_t)col * ng + gi] : T(0);
            }
#pragma unroll
        for (int t = 0; t < GT; ++t) {
            const int cb = c0 + 16 * t;
            if (cb < ncol) {  // uniform
#pragma unroll
                for (int jj = 0; jj < 16; jj += NC) {
                    const T re = gv[t][jj];
                    T im = T(0);
                    if constexpr (NC == 2) im = gv[t][jj + 1];
                    if constexpr (NC == 2) {
                        if constexpr (PH) {
                            stage[wave][lane][jj] = cs * re - sn * im;
                            stage[wave][lane][jj + 1] = cs * im + sn * re;
                        } else {
                            stage[wave][lane][jj] = re;
                            stage[wave][lane][jj + 1] = im;
                        }
                    } else {
                        stage[wave][lane][jj] = re;
                    }
                }
                // the stage is written and read by this wave only: its LDS
                // operations complete in order, and the fence keeps the
                // compiler from moving them across
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
                for (int s = 0; s < PJ_SUB / 4; ++s) {
                    const T b = stage[wave][4 * s + g][j];  // B[k = g][col = j]
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = M::mma(av[mt][s], b, acc[t][mt]);
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            }
        }
    }
    // sum of the four waves, tile by tile, in a fixed order
#pragma unroll
    for (int t = 0; t < GT; ++t) {
        const int cb = c0 + 16 * t;
        if (cb >= ncol) break;  // uniform over the workgroup
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][M::row(g, r) * 16 + j] = (double)acc[t][mt][r];
            __syncthreads();
            {
                const int e = threadIdx.x;  // 256 = 16 projectors x 16 columns
                const int w = e >> 4, cl = e & 15;
                if (cb + cl < ncol) {
                    const double sum = (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
                    part[((int64_t)item * MPAD + 16 * mt + w) * ncol + cb + cl] = sum;
                }
            }
            __syncthreads();
        }
    }
}

// tabp[v * mpad + w] = table of v's atom, projector w; zero past its projectors.
// From the tables already on the device: on the host, with the copy of both
// precisions, it was three quarters of setting a projector set (128 atoms, 2
// million voxels: 0.42 s of host time before the copy of 0.39 GB).
template <typename T>
__global__ void nl_padded_table_kernel(T *__restrict__ tabp, const T *__restrict__ table, int64_t n, int mpad,
                                       const int *__restrict__ vox_atom, const int64_t *__restrict__ vox_off,
                                       const int64_t *__restrict__ tab_off, const int *__restrict__ nproj) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int64_t v = e / mpad;
    const int w = (int)(e - v * mpad), a = vox_atom[v];
    const int64_t v0 = vox_off[a], V = vox_off[a + 1] - v0;
    tabp[e] = w < nproj[a] ? table[tab_off[a] + w * V + (v - v0)] : T(0);
}

// coef[p * ncol + col] = E_p dV sum over the atom's chunks (fixed order, FP64).
// Few threads, each with a chain of ~20 loads: latency bounds it, so kCoefLoads
// of them are requested together and added in chunk order (64^3 x 128, 16
// atoms: the FP32 nonlocal apply 97.6 -> 93.7 us, 32^3 x 24 FP64 20.7 -> 17.4).
constexpr int kCoefLoads = 8;
template <typename T>
__global__ void nl_coef_kernel(T *__restrict__ coef, const double *__restrict__ part, int ncol, int ptot, int mpad,
                               const int *__restrict__ proj_atom, const int *__restrict__ proj_off,
                               const int *__restrict__ atom_chunk_off, const double *__restrict__ energy, double dV) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= (int64_t)ptot * ncol) return;
    const int p = (int)(e / ncol), col = (int)(e % ncol);
    const int a = proj_atom[p];
    const int w = p - proj_off[a];
    const int it0 = atom_chunk_off[a], it1 = atom_chunk_off[a + 1];
    const double *src = part + (int64_t)w * ncol + col;
    const int64_t step = (int64_t)mpad * ncol;
    double s = 0.0;
    for (int it = it0; it < it1; it += kCoefLoads) {
        double v[kCoefLoads];
#pragma unroll
        for (int u = 0; u < kCoefLoads; ++u) v[u] = src[min(it + u, it1 - 1) * step];
#pragma unroll
        for (int u = 0; u < kCoefLoads; ++u)
            if (it + u < it1) s += v[u];
    }
    coef[e] = (T)(s * dV * energy[p]);
}

// Hpsi[col][g] += sum over (atom, voxel) entries covering g of (e^{-ik.r} sum_w p_w c_w)_col
// for the NG = NBS x GT real columns (NBS a multiple of NC) of column group
// g (logical block = point block * groups + g).  The coefficients of the (up to kScatterSlots) atoms a workgroup
// touches are staged in LDS; each thread reads its point's entry list and
// table rows once for the whole group.  MP: projector slots per entry (9 when
// every atom has at most 9 projectors, l <= 2, else the table padding of 16).
template <typename T, int NC, bool PH, int NBS, int GT, int MP>
__global__ __launch_bounds__(kScatterBlock) void nl_scatter_kernel(
    T *__restrict__ hpsi, const T *__restrict__ coef, int64_t ng, int ncol, int ncov,
    const int *__restrict__ cov_grid, const int *__restrict__ cov_off, const int *__restrict__ cov_vox,
    const int *__restrict__ cov_slot, const int *__restrict__ block_atom_off, const int *__restrict__ block_atoms,
    const int *__restrict__ vox_atom, const int *__restrict__ nproj, const int *__restrict__ proj_off,
    const T *__restrict__ tabp, const T *__restrict__ phase, int groups, int nblk, int per_xcd) {
    constexpr int NG = NBS * GT;  // columns of the group
    constexpr int MS = 16;  // table row padding
    __shared__ T cf_s[kScatterSlots][MP][NG];
    const int lb = xcd_block(nblk, per_xcd);
    if (lb < 0) return;  // the whole workgroup
    const int pb = lb / groups;  // point block
    const int cg = (lb - pb * groups) * NG;
    {
        const int b0 = block_atom_off[pb], nat = block_atom_off[pb + 1] - b0;
        for (int e = threadIdx.x; e < nat * MP * NG; e += kScatterBlock) {
            const int sl = e / (MP * NG), w = (e / NG) % MP, q = e % NG;
            const int a = block_atoms[b0 + sl];
            cf_s[sl][w][q] = (w < nproj[a] && cg + q < ncol) ? coef[(int64_t)(proj_off[a] + w) * ncol + cg + q] : T(0);
        }
    }
    __syncthreads();
    const int i = pb * kScatterBlock + threadIdx.x;
    if (i >= ncov) return;
    const int g = cov_grid[i];
    const int e0 = cov_off[i], e1 = cov_off[i + 1];  // e1 > e0: a covered point has an entry
    // An entry's voxel, slot, table row and phase are requested before the
    // point's NG values: the table row depends on the voxel index, so this
    // dependent round trip overlaps the NG loads instead of following them.
    int vid = cov_vox[e0], sl = cov_slot[e0];
    T pw[MP];
#pragma unroll
    for (int w = 0; w < MP; ++w) pw[w] = tabp[(int64_t)vid * MS + w];
    T cs = T(1), sn = T(0);
    if constexpr (PH) {
        cs = phase[2 * (int64_t)vid];
        sn = phase[2 * (int64_t)vid + 1];
    }
    // the point's values of all NG columns, requested together, then updated
    // in registers and written back once
    T hv[NG];
#pragma unroll
    for (int q = 0; q < NG; ++q) hv[q] = cg + q < ncol ? hpsi[(int64_t)(cg + q) * ng + g] : T(0);
    for (int e = e0;;) {
        if (sl >= 0) {
#pragma unroll
            for (int q = 0; q < NG; q += NC) {
                T tr = T(0), ti = T(0);
#pragma unroll
                for (int w = 0; w < MP; ++w) {
                    tr += pw[w] * cf_s[sl][w][q];
                    if constexpr (NC == 2) ti += pw[w] * cf_s[sl][w][q + 1];
                }
                if constexpr (PH) {
                    hv[q] += cs * tr + sn * ti;
                    hv[q + 1] += cs * ti - sn * tr;
                } else {
                    hv[q] += tr;
                    if constexpr (NC == 2) hv[q + 1] += ti;
                }
            }
        } else {  // more atoms in this workgroup than LDS slots: coefficients from global memory
            const int a = vox_atom[vid];
            const int M = nproj[a];
            const T *cf = coef + (int64_t)proj_off[a] * ncol + cg;
#pragma unroll
            for (int q = 0; q < NG; q += NC) {
                T tr = T(0), ti = T(0);
                if (cg + q < ncol) {
                    for (int w = 0; w < M; ++w) {
                        tr += pw[w] * cf[(int64_t)w * ncol + q];
                        if constexpr (NC == 2) ti += pw[w] * cf[(int64_t)w * ncol + q + 1];
                    }
                }
                if constexpr (PH) {
                    hv[q] += cs * tr + sn * ti;
                    hv[q + 1] += cs * ti - sn * tr;
                } else {
                    hv[q] += tr;
                    if constexpr (NC == 2) hv[q + 1] += ti;
                }
            }
        }
        if (++e >= e1) break;
        vid = cov_vox[e];
        sl = cov_slot[e];
#pragma unroll
        for (int w = 0; w < MP; ++w) pw[w] = tabp[(int64_t)vid * MS + w];
        if constexpr (PH) {
            cs = phase[2 * (int64_t)vid];
            sn = phase[2 * (int64_t)vid + 1];
        }
    }
#pragma unroll
    for (int q = 0; q < NG; ++q)
        if (cg + q < ncol) hpsi[(int64_t)(cg + q) * ng + g] = hv[q];
}

// The same sums on the matrix cores, for many projectors and small launches, where
// nl_scatter_kernel is bound by its broadcast LDS reads of the
// coefficients (one per point, column and projector).  A wave owns 16 PT
// covered points x 16 CT columns and takes the atoms of its tile one after the
// other: columns are the rows of the result (A: coefficients), points its
// columns (B: table rows) and projectors K, so each coefficient and table
// value is read once per 16 x 16 outputs.  K may run in any order: lane group q takes
// projectors KS q .. KS q + KS - 1, consecutive in the table row (KS: steps of
// 4 projectors; rows MS values apart).  A lane's 4 results are 4 consecutive
// columns in either precision (re and im of a band together, for the phase);
// an atom's results are added only at the points its sphere covers.  The sums
// then change lanes through LDS, so that Hpsi is read and written with lanes
// along the points (without it 64^3 x 64 complex took 110 us instead of 95).
// 45x54x50 x 37 complex FP64, 32 projectors, 45 -> 29 us (FP32 34 -> 22; 64^3 x 128
// FP32 116 -> 82); 32^3 x 24 FP64 6.5 -> 5.2 us.  Large launches with up to 9
// projectors are bound by Hpsi's lines (64^3 x 128 FP64: 0.41 GB of them in 97 us,
// 4.2 TB/s; 106 us here) and stay with nl_scatter_kernel, as does FP32 up to 16
// (half the LDS bytes a coefficient, and 32 columns a thread: 64^3 x 128 53 us
// there, 61 here; 160^3 x 512 3.19 and 3.41 ms).
template <typename T, int NC, bool PH, int KS, int CT, int PT>
__global__ __launch_bounds__(256) void nl_scatter_mfma_kernel(
    T *__restrict__ hpsi, const T *__restrict__ coef, int64_t ng, int ncol, int ntile,
    const int *__restrict__ cov_grid, const int *__restrict__ tile_row_off, const int *__restrict__ row_atom,
    const int *__restrict__ tile_vox, const int *__restrict__ nproj, const int *__restrict__ proj_off,
    const T *__restrict__ tabp, const T *__restrict__ phase, int groups, int nblk,
    int per_xcd) {
    using M = Mfma<T>;
    using acc_t = typename M::acc_t;
    constexpr int MS = KS > 4 ? 32 : 16;
    constexpr int SUBS = 4 / PT;               // waves per tile
    constexpr int P = 16 * PT, NV = CT * 4 * PT;  // a wave's points; values a lane moves
    __shared__ T stage[4][16 * CT][P + 16 / (int)sizeof(T)];
    const int lb = xcd_block(nblk, per_xcd);
    if (lb < 0) return;
    const int pb = lb / groups;
    const int cg = (lb - pb * groups) * 16 * CT;
    const int wave = threadIdx.x >> 6;
    const int sub = __builtin_amdgcn_readfirstlane(pb * 4 + wave);
    const int tile = sub / SUBS, t0 = (sub % SUBS) * PT;
    if (tile >= ntile) return;  // the whole wave
    const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
    // result row i of A holds column 4 (row's lane group) + (its item)
    const int ai = sizeof(T) == 8 ? 4 * (j & 3) + (j >> 2) : j;
    const int r0 = tile_row_off[tile], r1 = tile_row_off[tile + 1];  // r1 > r0: a covered point has an entry
    // the values of Hpsi are read and written with lanes along the points
    const int mp = lane & (P - 1), mc = lane / P;
    const int gi = cov_grid[tile * kScatterTile + 16 * t0 + mp];
    int vid[PT];
    T a[CT][KS], b[PT][KS];
    T cs[PT], sn[PT];
    // one row's voxels, coefficients, table rows and phases
    auto load_row = [&](int r) {
        const int at = row_atom[r], po = proj_off[at], np = nproj[at];
        const int *tv = tile_vox + (int64_t)r * kScatterTile + 4 * j + t0;
#pragma unroll
        for (int t = 0; t < PT; ++t) vid[t] = tv[t];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int col = cg + 16 * ct + ai;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int w = KS * q + s;
                a[ct][s] = (w < np && col < ncol) ? coef[(int64_t)(po + w) * ncol + col] : T(0);
            }
        }
#pragma unroll
        for (int t = 0; t < PT; ++t) {
            const int64_t v = max(vid[t], 0);
            const T *tr = tabp + v * MS + KS * q;
#pragma unroll
            for (int s = 0; s < KS; ++s) b[t][s] = tr[s];
            if constexpr (PH) {
                cs[t] = phase[2 * v];
                sn[t] = phase[2 * v + 1];
            }
        }
    };
    load_row(r0);
    // requested behind the first row's operands, which the first products wait for
    T *hp = hpsi + (int64_t)(cg + mc) * ng + max(gi, 0);
    T hv[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u)
        hv[u] = cg + mc + u * (64 / P) < ncol ? hp[(int64_t)u * (64 / P) * ng] : T(0);
    T sum[PT][CT][4];
#pragma unroll
    for (int t = 0; t < PT; ++t)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[t][ct][e] = T(0);
    for (int r = r0;;) {
#pragma unroll
        for (int t = 0; t < PT; ++t) {
            if (__ballot(vid[t] >= 0) == 0) continue;  // uniform
            acc_t acc[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                acc[ct] = acc_t{0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < KS; ++s) acc[ct] = M::mma(a[ct][s], b[t][s], acc[ct]);
            }
            // the table row behind a negative voxel is another point's: its
            // sums stay in their own column and are not added
            if (vid[t] >= 0) {
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int e = 0; e < 4; e += NC) {
                        if constexpr (PH) {
                            sum[t][ct][e] += cs[t] * acc[ct][e] + sn[t] * acc[ct][e + 1];
                            sum[t][ct][e + 1] += cs[t] * acc[ct][e + 1] - sn[t] * acc[ct][e];
                        } else {
                            sum[t][ct][e] += acc[ct][e];
                            if constexpr (NC == 2) sum[t][ct][e + 1] += acc[ct][e + 1];
                        }
                    }
            }
        }
        if (++r >= r1) break;
        load_row(r);
    }
    // the sums change lanes through the wave's own LDS slice
#pragma unroll
    for (int t = 0; t < PT; ++t)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e) stage[wave][16 * ct + 4 * q + e][16 * t + j] = sum[t][ct][e];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (gi < 0) return;
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (cg + mc + u * (64 / P) < ncol)
            hp[(int64_t)u * (64 / P) * ng] = hv[u] + stage[wave][mc + u * (64 / P)][mp];
}

// ---- forces -------------------------------------------------------------
// E_nl and F_a = 2 sum occ E Re(conj(<p|psi>) <dp/dr|psi>) need four projections
// per projector: by the table and by its three gradient tables.  They run as
// one projection with 4 max_m rows per atom (row q max_m + w: table q of
// projector w) in MT MFMA row tiles over the same voxel chunks as
// nl_project_kernel, so a psi value is gathered once for all four tables and
// the tables are read once per 16 columns.  Bound by the gather's latency, as
// the projection is.  64^3, 64 real FP64 bands, 8 atoms with 9 projectors: the
// earlier form (one workgroup per atom and band, 36 VALU accumulators a thread,
// every table re-read for every band) took 113 us; density + forces as one
// caller's sequence went from 206 to 90 us with this one.
//
// The tables are the caller's column-major ones (V_a values per row), so lane
// group g takes the 16 consecutive voxels 16 g .. 16 g + 15 of a 64-voxel
// sub-chunk: a lane's A operands of 16 K steps are then contiguous, and the
// K order of the sum is free as long as A and B agree on it.
//
// FP32 bands are summed on the FP64 matrix cores too: a wave's 128 voxels in one
// FP32 chain lost up to ten times what the earlier form's FP64 sum over threads
// did (bands of one sign, 4 atoms, forces: 3.6e-6 of the largest one, 5.4e-7 so).
// The gather hides the slower products: 64 real bands, 8 atoms 47.8 -> 49.7 us,
// 96^3, 64 complex bands, 40 atoms with 32 projectors 424 -> 443 us a call.

// Column slice of one launch and the occupations of its bands, by value: no
// staging buffer, no upload.
constexpr int kForceBands = 128;
struct ForceOcc {
    double occ[kForceBands];
};

// AS consecutive table values from p (aligned to T only)
template <typename T, int AS>
__device__ __forceinline__ void load_row(T (&out)[AS], const T *__restrict__ p) {
    typedef T vec_t __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
    constexpr int VEC = 16 / sizeof(T);
#pragma unroll
    for (int i = 0; i < AS; i += VEC) {
        const vec_t v = *reinterpret_cast<const vec_t *>(p + i);
#pragma unroll
        for (int c = 0; c < VEC; ++c) out[i + c] = v[c];
    }
}

// part[(item * 16 MT + r) * ncol + col]: row r of the item's voxels (see above)
// for the 16 columns of group g (logical block = item slot * groups + g).
template <typename T, int NC, bool PH, int MT>
__global__ __launch_bounds__(256) void nl_grad_project_kernel(
    double *__restrict__ part, const T *__restrict__ psi, int64_t ng, int ncol, int mm,
    const int *__restrict__ chunk_atom, const int *__restrict__ chunk_v0, const int64_t *__restrict__ vox_off,
    const int64_t *__restrict__ tab_off, int64_t ttot, const int *__restrict__ nproj,
    const int *__restrict__ vox_grid, const T *__restrict__ table, const T *__restrict__ dtable,
    const T *__restrict__ phase, const int *__restrict__ item_order, int groups, int nblk, int per_xcd) {
    constexpr int AS = MT == 1 ? 16 : (MT <= 4 ? 8 : 4);  // K steps whose A operands are held at once
    using M = Mfma<double>;
    using acc_t = typename M::acc_t;
    __shared__ T stage[4][PJ_SUB][16 + 1];
    __shared__ double red[4][16 * 16];
    const int lb = xcd_block(nblk, per_xcd);
    if (lb < 0) return;  // the whole workgroup
    const int slot = lb / groups;
    const int item = item_order[slot];
    const int c0 = (lb - slot * groups) * 16;
    const int a = chunk_atom[item];
    const int64_t vg0 = vox_off[a];
    const int V = (int)(vox_off[a + 1] - vg0);
    const int na = nproj[a];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int j = lane & 15, g = lane >> 4;
    const int vb = chunk_v0[item] + wave * PJ_VPW;
    // the lane's table row of each tile (row 0 of the table, unused, where there is none)
    const T *row[MT];
    bool has[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int r = 16 * mt + j, q = r / mm, w = r - q * mm;
        has[mt] = q < 4 && w < na;
        row[mt] = has[mt] && q > 0 ? dtable + (q - 1) * ttot + tab_off[a] + (int64_t)w * V
                                   : table + tab_off[a] + (has[mt] ? (int64_t)w * V : 0);
    }
    acc_t acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = acc_t{0, 0, 0, 0};
    for (int sc = 0; sc < PJ_VPW / PJ_SUB; ++sc) {
        const int vs = vb + sc * PJ_SUB;
        if (vs >= V) break;  // wave-uniform
        const int v = vs + lane;
        const bool in = v < V;
        const int64_t vid = vg0 + (in ? v : 0);
        const int gi = in ? vox_grid[vid] : 0;
        T cs = T(1), sn = T(0);
        if constexpr (PH) {
            cs = phase[2 * vid];
            sn = phase[2 * vid + 1];
        }
        T gv[16];
#pragma unroll
        for (int jj = 0; jj < 16; ++jj)
            gv[jj] = (in && c0 + jj < ncol) ? psi[(int64_t)(c0 + jj) * ng + gi] : T(0);
#pragma unroll
        for (int jj = 0; jj < 16; jj += NC) {
            const T re = gv[jj];
            if constexpr (NC == 2) {
                const T im = gv[jj + 1];
                stage[wave][lane][jj] = PH ? cs * re - sn * im : re;
                stage[wave][lane][jj + 1] = PH ? cs * im + sn * re : im;
            } else {
                stage[wave][lane][jj] = re;
            }
        }
        // written and read by this wave only (see nl_project_kernel)
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const bool whole = vs + PJ_SUB <= V && na > 0;  // wave-uniform: every row holds the sub-chunk's 64 values
#pragma unroll
        for (int h = 0; h < 16; h += AS) {
            T av[MT][AS];
            if (whole) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    load_row<T, AS>(av[mt], row[mt] + vs + 16 * g + h);
#pragma unroll
                    for (int s = 0; s < AS; ++s) av[mt][s] = has[mt] ? av[mt][s] : T(0);
                }
            } else {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int s = 0; s < AS; ++s) {
                        const int vv = vs + 16 * g + h + s;
                        av[mt][s] = has[mt] && vv < V ? row[mt][vv] : T(0);
                    }
            }
#pragma unroll
            for (int s = 0; s < AS; ++s) {
                const double b = (double)stage[wave][16 * g + h + s][j];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt] = M::mma((double)av[mt][s], b, acc[mt]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    // sum of the four waves in a fixed order
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][M::row(g, r) * 16 + j] = acc[mt][r];
        __syncthreads();
        const int e = threadIdx.x;  // 256 = 16 rows x 16 columns
        const int r = 16 * mt + (e >> 4), col = c0 + (e & 15);
        if (col < ncol && r < 4 * mm)
            part[((int64_t)item * (16 * MT) + r) * ncol + col] =
                (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
        __syncthreads();
    }
}

// Per (atom a, group of 16 columns): the chunk partials summed in order, then
// out[(blockIdx.y * natoms + a) * 4 + {0: E, 1..3: F}] over the group's bands.
// rows = 16 MT, mm = max_m.
template <int NC>
__global__ __launch_bounds__(256) void nl_force_sum_kernel(double *__restrict__ out, const double *__restrict__ part,
                                                           int ncol, int natoms, int mm, int rows, ForceOcc occ,
                                                           const int *__restrict__ atom_chunk_off,
                                                           const int *__restrict__ nproj,
                                                           const int *__restrict__ proj_off,
                                                           const double *__restrict__ energy, double dV) {
    __shared__ double S[4 * kMaxProj][16];
    __shared__ double red[4][4];
    const int a = blockIdx.x, c0 = blockIdx.y * 16;
    const int it0 = atom_chunk_off[a], it1 = atom_chunk_off[a + 1];
    const int64_t step = (int64_t)rows * ncol;
    for (int e = threadIdx.x; e < 4 * mm * 16; e += 256) {
        const int r = e >> 4, cl = e & 15;
        double s = 0.0;
        if (c0 + cl < ncol) {
            const double *src = part + (int64_t)r * ncol + c0 + cl;
            for (int it = it0; it < it1; it += kCoefLoads) {
                double v[kCoefLoads];
#pragma unroll
                for (int u = 0; u < kCoefLoads; ++u) v[u] = src[min(it + u, it1 - 1) * step];
#pragma unroll
                for (int u = 0; u < kCoefLoads; ++u)
                    if (it + u < it1) s += v[u];
            }
        }
        S[r][cl] = s * dV;
    }
    __syncthreads();
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    const int M = nproj[a];
    for (int e = threadIdx.x; e < M * (16 / NC); e += 256) {
        const int b = e / M, w = e - b * M;
        const int cl = b * NC;
        if (c0 + cl >= ncol) break;  // columns past the slice hold no band
        const double eo = energy[proj_off[a] + w] * occ.occ[(c0 + cl) / NC];
        const double pr = S[w][cl], pi = NC == 2 ? S[w][cl + NC - 1] : 0.0;
        t[0] += (pr * pr + pi * pi) * eo;
#pragma unroll
        for (int d = 1; d < 4; ++d) {
            const double gr = S[d * mm + w][cl], gim = NC == 2 ? S[d * mm + w][cl + NC - 1] : 0.0;
            t[d] += 2.0 * (pr * gr + pi * gim) * eo;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const double s = wave_sum<double>(t[d]);
        if (lane == 0) red[wave][d] = s;
    }
    __syncthreads();
    if (threadIdx.x < 4)
        out[((int64_t)blockIdx.y * natoms + a) * 4 + threadIdx.x] =
            (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
}

template <typename T>
const T *table_of(const Projectors &p);
template <>
const double *table_of<double>(const Projectors &p) { return p.d_table64; }
template <>
const float *table_of<float>(const Projectors &p) { return p.d_table32; }
template <typename T>
const T *dtable_of(const Projectors &p);
template <>
const double *dtable_of<double>(const Projectors &p) { return p.d_dtable64; }
template <>
const float *dtable_of<float>(const Projectors &p) { return p.d_dtable32; }
template <typename T>
const T *phase_of(const KPoint &k);
template <>
const double *phase_of<double>(const KPoint &k) { return k.d_phase64; }
template <>
const float *phase_of<float>(const KPoint &k) { return k.d_phase32; }

template <typename T>
const T *tabp_of(const Projectors &p);
template <>
const double *tabp_of<double>(const Projectors &p) { return p.d_tabp_64; }
template <>
const float *tabp_of<float>(const Projectors &p) { return p.d_tabp_32; }

constexpr int64_t kProjMinBlocks = 1024;  // 4 workgroups per CU

// Tuning key of a projection shape; band counts share a key within a
// power-of-two bucket (as the stencil's).
int64_t nl_tune_key(int precision, int nc, bool ph, int mpad, int nb) {
    int64_t bucket = 1;
    while (bucket < nb) bucket <<= 1;
    return ((((bucket * 4 + (nc - 1) * 2 + (ph ? 1 : 0)) * 64) + mpad) << 8) | precision;
}

template <typename T, int NC, bool PH, int GT, int MT>
void launch_project(qm_ctx *ctx, double *part, const T *psi, int ncol, const T *phase, hipStream_t st) {
    const Projectors &p = ctx->proj;
    const int groups = (ncol + 16 * GT - 1) / (16 * GT);
    const int64_t nblk = (int64_t)p.nchunk * groups;
    const int per_xcd = (int)((nblk + 7) / 8);
    hipLaunchKernelGGL((nl_project_kernel<T, NC, PH, GT, MT>), dim3(8 * per_xcd), dim3(256), 0, st, part, psi, ctx->ng,
                       ncol, p.d_chunk_atom, p.d_chunk_v0, p.d_vox_off, p.d_vox_grid, tabp_of<T>(p), phase,
                       p.d_item_order, groups, (int)nblk, per_xcd);
}

// Projection coefficients of nb bands into coef (ptot x ncol, T) through the
// per-chunk partial sums part (nchunk x mpad x ncol, FP64).  Both buffers
// are written in full before they are read, so they need no clearing.
template <typename T, int NC, bool PH>
int nonlocal_project(qm_ctx *ctx, T *coef, double *part, const T *psi, int nb, const T *phase, hipStream_t st) {
    const Projectors &p = ctx->proj;
    const int ncol = nb * NC;
    // 4 tiles of 16 columns per projection workgroup share each table read;
    // the columns beyond split over more workgroups.  A launch that would then
    // have fewer than kProjMinBlocks workgroups (a small grid or few bands:
    // 64^3 x 128 has 640) takes 1 tile per workgroup instead, for four times
    // the workgroups in flight on this latency-bound gather (2 tiles measured
    // 1-2 % slower there).  Each column's sum runs over the same voxels in the
    // same order either way, so every shape gives the same values.  The first
    // projection of a shape (precision, ncomp, phases, padding, band-count
    // bucket) times the candidates on the caller's buffers (the projection only
    // writes its own partial sums) and keeps the fastest; tables padded to 32
    // projectors (two MFMA row tiles per table read) take at most 2 column
    // tiles, for the registers.
    const int64_t g4 = (ncol + 63) / 64;
    QM_CHECK((int64_t)p.nchunk * g4 * 4 < (int64_t)INT32_MAX / 16, QM_ERR_ARG,
             "nonlocal apply: too many bands per call");
    auto launch = [&](int gt) {
        if (p.mpad == 16) {
            if (gt == 4) launch_project<T, NC, PH, 4, 1>(ctx, part, psi, ncol, phase, st);
            else if (gt == 2) launch_project<T, NC, PH, 2, 1>(ctx, part, psi, ncol, phase, st);
            else launch_project<T, NC, PH, 1, 1>(ctx, part, psi, ncol, phase, st);
        } else {
            if (gt >= 2) launch_project<T, NC, PH, 2, 2>(ctx, part, psi, ncol, phase, st);
            else launch_project<T, NC, PH, 1, 2>(ctx, part, psi, ncol, phase, st);
        }
    };
    const int max_gt = p.mpad == 16 ? 4 : 2;
    int gt = ctx->nl_force > 0 ? std::min(ctx->nl_force, max_gt) : 0;
    if (gt == 0) {
        const int64_t key = nl_tune_key(sizeof(T) == 8 ? 64 : 32, NC, PH, p.mpad, nb);
        auto it = ctx->nl_choice.find(key);
        if (it != ctx->nl_choice.end()) {
            gt = it->second;
        } else {
            hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
            QM_HIP(hipStreamIsCapturing(st, &cs));
            if (cs != hipStreamCaptureStatusNone || g_internal_capture || ctx->nl_notime) {
                gt = (int64_t)p.nchunk * g4 >= kProjMinBlocks ? max_gt : 1;  // no timing inside a capture
            } else {
                hipEvent_t ev[2] = {nullptr, nullptr};
                QM_HIP(hipEventCreate(&ev[0]));
                if (hipEventCreate(&ev[1]) != hipSuccess) {
                    (void)hipEventDestroy(ev[0]);
                    QM_CHECK(false, QM_ERR_HIP, "nonlocal autotune: hipEventCreate failed");
                }
                float best = 1e30f;
                int status = QM_OK;
                for (int cand = 1; cand <= max_gt && status == QM_OK; cand *= 2) {
                    launch(cand);  // warm-up
                    float ms = 0.0f;
                    if (hipEventRecord(ev[0], st) != hipSuccess) status = QM_ERR_HIP;
                    for (int rep = 0; rep < 3 && status == QM_OK; ++rep) launch(cand);
                    if (status == QM_OK && hipEventRecord(ev[1], st) != hipSuccess) status = QM_ERR_HIP;
                    if (status == QM_OK && hipEventSynchronize(ev[1]) != hipSuccess) status = QM_ERR_HIP;
                    if (status == QM_OK && hipEventElapsedTime(&ms, ev[0], ev[1]) != hipSuccess) status = QM_ERR_HIP;
                    if (status == QM_OK && hipGetLastError() != hipSuccess) status = QM_ERR_HIP;
                    if (status == QM_OK && ms < best) {
                        best = ms;
                        gt = cand;
                    }
                }
                (void)hipEventDestroy(ev[0]);
                (void)hipEventDestroy(ev[1]);
                QM_CHECK(status == QM_OK, QM_ERR_HIP, "nonlocal autotune: HIP failure");
                ctx->nl_choice[key] = gt;
            }
        }
    }
    launch(gt);
    QM_HIP(hipGetLastError());
    const int64_t ncoef = (int64_t)p.ptot * ncol;
    hipLaunchKernelGGL((nl_coef_kernel<T>), dim3((unsigned)((ncoef + 255) / 256)), dim3(256), 0, st, coef, part, ncol,
                       p.ptot, p.mpad, p.d_proj_atom, p.d_proj_off, p.d_atom_chunk_off, p.d_energy,
                       ctx->hx * ctx->hy * ctx->hz);
    QM_HIP(hipGetLastError());
    return QM_OK;
}

template <typename T, int NC, bool PH, int KS, int CT, int PT>
int launch_scatter_mfma(qm_ctx *ctx, T *hpsi, const T *coef, int ncol, const T *phase, hipStream_t st) {
    const Projectors &p = ctx->proj;
    const int groups = (ncol + 16 * CT - 1) / (16 * CT);
    const int64_t nblk = (int64_t)((p.ntile + PT - 1) / PT) * groups;
    QM_CHECK(nblk < (int64_t)INT32_MAX / 16, QM_ERR_ARG, "nonlocal apply: too many bands per call");
    const int per_xcd = (int)((nblk + 7) / 8);
    hipLaunchKernelGGL((nl_scatter_mfma_kernel<T, NC, PH, KS, CT, PT>), dim3(8 * per_xcd), dim3(256), 0, st, hpsi,
                       coef, ctx->ng, ncol, p.ntile, p.d_cov_grid, p.d_tile_row_off, p.d_row_atom, p.d_tile_vox,
                       p.d_nproj, p.d_proj_off, tabp_of<T>(p), phase, groups, (int)nblk, per_xcd);
    QM_HIP(hipGetLastError());
    return QM_OK;
}

// Waves of the MFMA scatter with 32 points x 32 columns each
inline int64_t scatter_waves(const Projectors &p, int ncol) { return (int64_t)p.ntile * 2 * ((ncol + 31) / 32); }

// 32 points x 32 columns a wave; 16 x 16 where that leaves less than 2 waves a
// SIMD (32^3 x 24 FP64: 576 waves 6.9 us, 2272 waves 5.2 us; 36x40x42 x 45
// complex: 3100 waves 21 us, 12400 waves 24 us)
template <typename T, int NC, bool PH, int KS>
int scatter_mfma(qm_ctx *ctx, T *hpsi, const T *coef, int ncol, const T *phase, hipStream_t st) {
    if (scatter_waves(ctx->proj, ncol) >= 2048)
        return launch_scatter_mfma<T, NC, PH, KS, 2, 2>(ctx, hpsi, coef, ncol, phase, st);
    return launch_scatter_mfma<T, NC, PH, KS, 1, 1>(ctx, hpsi, coef, ncol, phase, st);
}

// columns per scatter tile (16; 64 per thread measured 1.9x slower on 64^3 x
// 128) and tiles per workgroup (the staged coefficients, entry lists and table
// rows serve all of them)
template <typename T, int NC, bool PH, int MP>
int scatter_points(qm_ctx *ctx, T *hpsi, const T *coef, int ncol, const T *phase, hipStream_t st) {
    const Projectors &p = ctx->proj;
    constexpr int NBS = 16, SGT = sizeof(T) == 8 ? 1 : 2;
    const int sgroups = (ncol + NBS * SGT - 1) / (NBS * SGT);
    const int64_t nblk = (int64_t)p.nsblock * sgroups;
    QM_CHECK(nblk < (int64_t)INT32_MAX / 16, QM_ERR_ARG, "nonlocal apply: too many bands per call");
    const int per_xcd = (int)((nblk + 7) / 8);
    hipLaunchKernelGGL((nl_scatter_kernel<T, NC, PH, NBS, SGT, MP>), dim3(8 * per_xcd), dim3(kScatterBlock), 0, st,
                       hpsi, coef, ctx->ng, ncol, p.ncov, p.d_cov_grid, p.d_cov_off, p.d_cov_vox, p.d_cov_slot,
                       p.d_block_atom_off, p.d_block_atoms, p.d_vox_atom, p.d_nproj, p.d_proj_off, tabp_of<T>(p), phase,
                       sgroups, (int)nblk, per_xcd);
    QM_HIP(hipGetLastError());
    return QM_OK;
}

template <typename T, int NC, bool PH>
int nonlocal_scatter(qm_ctx *ctx, T *hpsi, const T *coef, int nb, const T *phase, hipStream_t st) {
    const int ncol = nb * NC, m = ctx->proj.max_m;
    if (m > 16) return scatter_mfma<T, NC, PH, 8>(ctx, hpsi, coef, ncol, phase, st);
    if constexpr (sizeof(T) == 8) {
        if (m > 12) return scatter_mfma<T, NC, PH, 4>(ctx, hpsi, coef, ncol, phase, st);
        // up to 9 projectors the thread-per-point kernel wins on large launches, not
        // with 16 (64^3 x 64 complex: 109 us there, 101 here).  40 applies timed both ways
        // (us here less us there): 560 - 3000 waves -1.8 .. -0.2 of 15 - 34; 4000 - 4500 real
        // +1.6 .. +2.6 of 43 - 50, complex -1.3 .. +0.1; 5200 - 8500 real -3.5 .. +6.2 of 53 -
        // 88 (10 of 12 above 0), complex -2.3 .. +2.4; 11,000 - 17,000 real +2.7 .. +11 of 116 -
        // 179, complex -0.3 .. +1.7
        if (m > 9 || scatter_waves(ctx->proj, ncol) < 4096)
            return scatter_mfma<T, NC, PH, 3>(ctx, hpsi, coef, ncol, phase, st);
        return scatter_points<T, NC, PH, 9>(ctx, hpsi, coef, ncol, phase, st);
    } else {
        if (m > 9) return scatter_points<T, NC, PH, 16>(ctx, hpsi, coef, ncol, phase, st);
        return scatter_points<T, NC, PH, 9>(ctx, hpsi, coef, ncol, phase, st);
    }
}

// which: 1 = projection coefficients, 2 = scatter, 3 = both.  coef / part are
// the work buffers (nonlocal_work_bytes); NULL takes the context's own, grown
// as needed.
template <typename T>
int launch_nonlocal(qm_ctx *ctx, T *hpsi, const T *psi, int nb, int ncomp, const KPoint &kp, hipStream_t st,
                    int which = 3, T *coef = nullptr, double *part = nullptr) {
    const Projectors &p = ctx->proj;
    if (p.natoms == 0 || p.ptot == 0) return QM_OK;
    const bool ph = !kp.gamma;
    QM_CHECK(ncomp == 2 || !ph, QM_ERR_ARG, "real (ncomp=1) bands need a Gamma k-point");
    const T *phase = phase_of<T>(kp);
    size_t cb = 0, pb = 0;
    nonlocal_work_bytes(ctx, nb, ncomp, sizeof(T), &cb, &pb);
    if (!coef && ctx->capture_pins) {  // a caller's graph holds the current work buffers
        QM_CHECK(ctx->coef.bytes >= cb && ((which & 1) == 0 || ctx->nl_part.bytes >= pb), QM_ERR_STATE,
                 "H.psi apply: larger nonlocal work buffers needed (more bands, or FP64 after FP32) while a "
                 "graph holds an apply of this context; destroy it and call qm_release_captures first");
    }
    if (!coef) {
        if (which & 1) QM_TRY(ctx->coef.reserve(cb));
        QM_CHECK(ctx->coef.bytes >= cb, QM_ERR_STATE,
                 "nonlocal scatter: no projection coefficients for this band count");
        coef = ctx->coef.as<T>();
    }
    if ((which & 1) && !part) {
        QM_TRY(ctx->nl_part.reserve(pb));
        part = ctx->nl_part.as<double>();
    }
    if (which & 1) {
        if (ncomp == 1) QM_TRY((nonlocal_project<T, 1, false>(ctx, coef, part, psi, nb, phase, st)));
        else if (!ph) QM_TRY((nonlocal_project<T, 2, false>(ctx, coef, part, psi, nb, phase, st)));
        else QM_TRY((nonlocal_project<T, 2, true>(ctx, coef, part, psi, nb, phase, st)));
    }
    if (which & 2) {
        if (ncomp == 1) QM_TRY((nonlocal_scatter<T, 1, false>(ctx, hpsi, coef, nb, phase, st)));
        else if (!ph) QM_TRY((nonlocal_scatter<T, 2, false>(ctx, hpsi, coef, nb, phase, st)));
        else QM_TRY((nonlocal_scatter<T, 2, true>(ctx, hpsi, coef, nb, phase, st)));
    }
    return QM_OK;
}

template <typename T, int NC, bool PH, int MT>
void launch_grad_project(qm_ctx *ctx, double *part, const T *psi, int ncol, const T *phase, hipStream_t st) {
    const Projectors &p = ctx->proj;
    const int groups = (ncol + 15) / 16;
    const int64_t nblk = (int64_t)p.nchunk * groups;
    const int per_xcd = (int)((nblk + 7) / 8);
    hipLaunchKernelGGL((nl_grad_project_kernel<T, NC, PH, MT>), dim3(8 * per_xcd), dim3(256), 0, st, part, psi,
                       ctx->ng, ncol, p.max_m, p.d_chunk_atom, p.d_chunk_v0, p.d_vox_off, p.d_tab_off, p.ttot,
                       p.d_nproj, p.d_vox_grid, table_of<T>(p), dtable_of<T>(p), phase, p.d_item_order, groups,
                       (int)nblk, per_xcd);
}

// One slice of bands: the projections, then the sums into out (groups x natoms x 4)
template <typename T, int NC, bool PH>
int launch_force(qm_ctx *ctx, double *out, double *part, int mt, const T *psi, int nb, const ForceOcc &occ,
                 const T *phase, hipStream_t st) {
    const Projectors &p = ctx->proj;
    const int ncol = nb * NC;
    switch (mt) {
        case 1: launch_grad_project<T, NC, PH, 1>(ctx, part, psi, ncol, phase, st); break;
        case 3: launch_grad_project<T, NC, PH, 3>(ctx, part, psi, ncol, phase, st); break;
        case 4: launch_grad_project<T, NC, PH, 4>(ctx, part, psi, ncol, phase, st); break;
        default: launch_grad_project<T, NC, PH, 8>(ctx, part, psi, ncol, phase, st); break;
    }
    QM_HIP(hipGetLastError());
    hipLaunchKernelGGL((nl_force_sum_kernel<NC>), dim3(p.natoms, (ncol + 15) / 16), dim3(256), 0, st, out, part, ncol,
                       p.natoms, p.max_m, 16 * mt, occ, p.d_atom_chunk_off, p.d_nproj, p.d_proj_off, p.d_energy,
                       ctx->hx * ctx->hy * ctx->hz);
    QM_HIP(hipGetLastError());
    return QM_OK;
}

constexpr int64_t kForcePartBytes = (int64_t)128 << 20;  // partial sums of one slice of bands

template <typename T>
int nonlocal_forces(qm_ctx *ctx, const T *psi, const double *occ, int nb, int ncomp, const KPoint &kp,
                    double *forces, double *e_nl, hipStream_t st) {
    const Projectors &p = ctx->proj;
    QM_CHECK(p.has_grad, QM_ERR_STATE, "nonlocal forces need the projector gradient tables (dtable)");
    QM_CHECK(ncomp == 1 || ncomp == 2, QM_ERR_ARG, "ncomp must be 1 or 2");
    const bool ph = !kp.gamma;
    QM_CHECK(ncomp == 2 || !ph, QM_ERR_ARG, "real (ncomp=1) bands need a Gamma k-point");
    *e_nl = 0.0;
    for (int i = 0; i < 3 * p.natoms; ++i) forces[i] = 0.0;
    if (p.nchunk == 0 || p.max_m == 0) {  // no voxels or no projectors: nothing to sum
        QM_HIP(hipStreamSynchronize(st));
        return QM_OK;
    }
    // MFMA row tiles of the 4 max_m projections (1, 3, 4 or 8 are built: up to
    // 4, 12, 16 and 32 projectors per atom)
    const int need = (4 * p.max_m + 15) / 16;
    const int mt = need <= 1 ? 1 : (need <= 3 ? 3 : (need == 4 ? 4 : 8));
    // bands per slice: what the partial sums' limit allows, in whole groups of
    // 16 columns, at most kForceBands
    const int64_t per_band = (int64_t)p.nchunk * 16 * mt * ncomp * (int64_t)sizeof(double);
    const int slice = (int)std::max<int64_t>(16, std::min<int64_t>(kForceBands, kForcePartBytes / per_band / 16 * 16));
    QM_CHECK((int64_t)p.nchunk * ((slice * ncomp + 15) / 16) < (int64_t)INT32_MAX / 16, QM_ERR_ARG,
             "nonlocal forces: too many projector voxels");
    const int gmax = (slice * ncomp + 15) / 16;  // column groups of a slice
    const int nslice = (nb + slice - 1) / slice;
    const size_t part_bytes = (size_t)per_band * std::min(slice, nb);
    const size_t out_n = (size_t)nslice * gmax * p.natoms * 4;
    QM_TRY(ctx->fwork.reserve(part_bytes));
    double *part = ctx->fwork.as<double>();
    // the kernels write the sums, four values per atom and 16 columns, into pinned
    // memory (density and forces of 64^3 x 64 FP64 bands, 8 atoms: 91 us with a
    // copy to pageable memory after them, 83 so)
    if (ctx->h_force_n < out_n) {
        if (ctx->h_force) (void)hipHostFree(ctx->h_force);
        ctx->h_force = nullptr;
        ctx->h_force_n = 0;
        QM_HIP(hipHostMalloc((void **)&ctx->h_force, sizeof(double) * out_n, hipHostMallocDefault));
        ctx->h_force_n = out_n;
    }
    const T *phase = phase_of<T>(kp);
    size_t used = 0;  // output blocks of 4 natoms values written so far
    for (int n0 = 0; n0 < nb; n0 += slice) {
        const int n = std::min(slice, nb - n0);
        ForceOcc fo;
        for (int i = 0; i < kForceBands; ++i) fo.occ[i] = i < n ? occ[n0 + i] : 0.0;
        double *out = ctx->h_force + used * p.natoms * 4;
        const T *src = psi + (int64_t)n0 * ncomp * ctx->ng;
        if (ncomp == 1) QM_TRY((launch_force<T, 1, false>(ctx, out, part, mt, src, n, fo, phase, st)));
        else if (!ph) QM_TRY((launch_force<T, 2, false>(ctx, out, part, mt, src, n, fo, phase, st)));
        else QM_TRY((launch_force<T, 2, true>(ctx, out, part, mt, src, n, fo, phase, st)));
        used += (n * ncomp + 15) / 16;
    }
    QM_HIP(hipStreamSynchronize(st));
    double e = 0.0;
    for (int a = 0; a < p.natoms; ++a)
        for (size_t g = 0; g < used; ++g) {
            const double *o4 = &ctx->h_force[(g * p.natoms + a) * 4];
            e += o4[0];
            for (int d = 0; d < 3; ++d) forces[3 * a + d] += o4[1 + d];
        }
    *e_nl = e;
    return QM_OK;
}

}  // namespace

int padded_tables(Projectors &p) {
    const int64_t n = p.vtot * p.mpad;
    if (n == 0) return QM_OK;
    const dim3 grid((unsigned)((n + 255) / 256));
    hipError_t e = hipMalloc((void **)&p.d_tabp_64, sizeof(double) * n);
    if (e == hipSuccess) e = hipMalloc((void **)&p.d_tabp_32, sizeof(float) * n);
    QM_CHECK(e == hipSuccess, QM_ERR_NOMEM, std::string("hipMalloc failed: ") + hipGetErrorString(e));
    hipLaunchKernelGGL(nl_padded_table_kernel<double>, grid, dim3(256), 0, nullptr, p.d_tabp_64, p.d_table64, n, p.mpad,
                       p.d_vox_atom, p.d_vox_off, p.d_tab_off, p.d_nproj);
    hipLaunchKernelGGL(nl_padded_table_kernel<float>, grid, dim3(256), 0, nullptr, p.d_tabp_32, p.d_table32, n, p.mpad,
                       p.d_vox_atom, p.d_vox_off, p.d_tab_off, p.d_nproj);
    QM_HIP(hipGetLastError());
    return QM_OK;
}

int launch_nonlocal_f64(qm_ctx *ctx, double *hpsi, const double *psi, int nb, int ncomp, const KPoint &kp,
                        hipStream_t st) {
    return launch_nonlocal<double>(ctx, hpsi, psi, nb, ncomp, kp, st);
}
int launch_nonlocal_f32(qm_ctx *ctx, float *hpsi, const float *psi, int nb, int ncomp, const KPoint &kp,
                        hipStream_t st) {
    return launch_nonlocal<float>(ctx, hpsi, psi, nb, ncomp, kp, st);
}
int nonlocal_project_f64(qm_ctx *ctx, const double *psi, int nb, int ncomp, const KPoint &kp, hipStream_t st) {
    return launch_nonlocal<double>(ctx, nullptr, psi, nb, ncomp, kp, st, 1);
}
int nonlocal_project_f32(qm_ctx *ctx, const float *psi, int nb, int ncomp, const KPoint &kp, hipStream_t st) {
    return launch_nonlocal<float>(ctx, nullptr, psi, nb, ncomp, kp, st, 1);
}
int nonlocal_scatter_f64(qm_ctx *ctx, double *hpsi, int nb, int ncomp, const KPoint &kp, hipStream_t st) {
    return launch_nonlocal<double>(ctx, hpsi, nullptr, nb, ncomp, kp, st, 2);
}
int nonlocal_scatter_f32(qm_ctx *ctx, float *hpsi, int nb, int ncomp, const KPoint &kp, hipStream_t st) {
    return launch_nonlocal<float>(ctx, hpsi, nullptr, nb, ncomp, kp, st, 2);
}
// Bytes of the two nonlocal work buffers for nb bands: the coefficients
// (ptot x ncol, T) and the per-chunk partial sums (nchunk x mpad x ncol, FP64).
void nonlocal_work_bytes(const qm_ctx *ctx, int nb, int ncomp, size_t tsize, size_t *coef_bytes,
                         size_t *part_bytes) {
    const Projectors &p = ctx->proj;
    const size_t ncol = (size_t)nb * ncomp;
    *coef_bytes = tsize * (size_t)p.ptot * ncol;
    *part_bytes = sizeof(double) * (size_t)p.nchunk * p.mpad * ncol;
}

int nonlocal_choice(const qm_ctx *ctx, int precision, int ncomp, int kt, int nb) {
    if (ctx->nl_force > 0) return ctx->nl_force;
    const int64_t key = nl_tune_key(precision, ncomp, (kt & 1) != 0 && ncomp == 2, ctx->proj.mpad, nb);
    auto it = ctx->nl_choice.find(key);
    return it == ctx->nl_choice.end() ? -1 : it->second;
}

int nonlocal_apply_in_f32(qm_ctx *ctx, float *hpsi, const float *psi, int nb, int ncomp, const KPoint &kp,
                          int which, float *coef, double *part, hipStream_t st) {
    return launch_nonlocal<float>(ctx, hpsi, psi, nb, ncomp, kp, st, which, coef, part);
}
int nonlocal_forces_f64(qm_ctx *ctx, const double *psi, const double *occ, int nb, int ncomp, const KPoint &kp,
                        double *forces, double *e_nl, hipStream_t st) {
    return nonlocal_forces<double>(ctx, psi, occ, nb, ncomp, kp, forces, e_nl, st);
}
int nonlocal_forces_f32(qm_ctx *ctx, const float *psi, const double *occ, int nb, int ncomp, const KPoint &kp,
                        double *forces, double *e_nl, hipStream_t st) {
    return nonlocal_forces<float>(ctx, psi, occ, nb, ncomp, kp, forces, e_nl, st);
}

}  // namespace qm
