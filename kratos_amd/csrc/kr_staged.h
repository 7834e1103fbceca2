// kr_staged.h -- the staged Godunov kernels: one launch per stage step, each
// launch covering every block of the mesh (grid.y = block), SoA state in
// HBM, neighbour-table reads instead of ghost copies.
//
// Per RK substep: k_c2p -> (k_dt_finalize at substep 0) -> k_flux x ndim
// -> k_emf (MHD) -> k_update.  This is the reference's integrate() pipeline
// (dynamics/dynamics.h:60-100) without per-block launches, streams, host
// syncs or halo-copy kernels.
#pragma once

#include "kr_mesh.h"
#include "kr_exact64.h"

namespace kr {

constexpr int kThreads = 256;

// ------------------------------------------------------------------ index
__device__ __forceinline__ size_t cidx(const int *n, int i, int j, int k) {
    return ((size_t)k * n[1] + j) * n[0] + i;
}
__device__ __forceinline__ size_t fidx(const int *n, int i, int j, int k) {
    return ((size_t)k * (n[1] + 1) + j) * (n[0] + 1) + i;
}
// flux box of sweep axis `ax`: n+1 faces along ax, n+2 (one ghost line on
// each side) along the transverse axes.
__device__ __forceinline__ size_t xidx(const int *n, int ax, const int *p) {
    const int d0 = n[0] + (ax == 0 ? 1 : 2), d1 = n[1] + (ax == 1 ? 1 : 2);
    const int o0 = ax == 0 ? 0 : 1, o1 = ax == 1 ? 0 : 1, o2 = ax == 2 ? 0 : 1;
    return ((size_t)(p[2] + o2) * d1 + (p[1] + o1)) * d0 + (p[0] + o0);
}

// Block handled by grid row blockIdx.y of a stage kernel.
template <class FT>
__device__ __forceinline__ int row_block(const MeshView<FT> &m) {
    return m.blist ? m.blist[blockIdx.y] : (int)blockIdx.y;
}

template <class FT>
__device__ __forceinline__ int nbr_dir(const MeshView<FT> &m, const int *d) {
    return ((d[2] + 1) * 3 + (d[1] + 1)) * 3 + (d[0] + 1);
}

// Where the primitives of a cell come from: cell p of block blk, then the
// boundary functor of a physical side.
struct CellSrc {
    int blk, p[3];
    int flip;       // axis of a reflecting side, -1: none
    int clamp;      // 2 * axis + side of an outflow side, -1: none
    bool fixd;      // Dirichlet side: the ghost is the fixed state
};

// Source of cell pin of block b.  Cells outside the block come from the
// same-level neighbour (the reference fills them by the ghost exchange,
// hydro/boundary/comm_functions.h:304-327); on a physical side the
// reference's boundary functor is applied on the fly
// (hydro/boundary/phys_functors.h:10-89).
template <class FT, int NV>
__device__ __forceinline__ CellSrc cell_src(const MeshView<FT> &m, int b, const int *pin) {
    CellSrc c;
    int p[3] = {pin[0], pin[1], pin[2]};
    int d[3];
    bool out = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        d[a] = p[a] < 0 ? -1 : (p[a] >= m.n[a] ? 1 : 0);
        out |= d[a] != 0;
    }
    c.blk = b;
    c.flip = -1;
    c.clamp = -1;
    c.fixd = false;
    if (out) {
        const int nb = m.geo[b].nbr[nbr_dir(m, d)];
        if (nb >= 0) {
            c.blk = nb;
#pragma unroll
            for (int a = 0; a < 3; ++a) p[a] -= d[a] * m.n[a];
        } else if constexpr (NV == 5) {
            // physical side: one axis out of range (hydro face ghosts);
            // every index below is resolved with unrolled selects so the
            // register arrays keep static indices.
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if (d[a] == 0) continue;
                const int side = d[a] > 0;
                const int kind = m.bnd[2 * a + side];
                const int g = side ? p[a] - m.n[a] : -1 - p[a];
                if (kind == 3) {                       // reflect
                    p[a] = side ? m.n[a] - 1 - g : g;
                    c.flip = a;
                } else {                               // outflow / free / fixd
                    p[a] = side ? m.n[a] - 1 : 0;
                    if (kind == 1) c.clamp = 2 * a + side;
                    if (kind == 4) c.fixd = true;
                }
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) p[a] = p[a] < 0 ? 0 : (p[a] >= m.n[a] ? m.n[a] - 1 : p[a]);
        } else {
            // MHD physical side (mhd/boundary/phys.h:144-251): the cell is
            // written last by the side of the highest out-of-range axis that
            // is physical; its source is mirrored (reflect) or the boundary
            // cell (free / outflow) along that axis, clamped into the block
            // along other axes that are physical on that end, and taken from
            // the neighbour along the remaining (periodic / internal) ones.
            const BlockGeo &g = m.geo[b];
            int al = 0;
#pragma unroll
            for (int a = 0; a < 3; ++a)
                if (d[a] != 0 && ((g.phy >> (2 * a + (d[a] > 0))) & 1)) al = a;
            int q[3], e[3];
            bool out2 = false;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int side = d[a] > 0;
                q[a] = p[a];
                if (a == al) {
                    const int kind = m.bnd[2 * a + side];
                    const int gd = side ? p[a] - m.n[a] : -1 - p[a];
                    if (kind == 3) {
                        q[a] = side ? m.n[a] - 1 - gd : gd;
                        c.flip = a;
                    } else {
                        q[a] = side ? m.n[a] - 1 : 0;
                        if (kind == 1) c.clamp = 2 * a + side;
                        if (kind == 4) c.fixd = true;
                    }
                } else if (d[a] != 0 && ((g.phy >> (2 * a + side)) & 1)) {
                    q[a] = side ? m.n[a] - 1 : 0;
                }
                e[a] = q[a] < 0 ? -1 : (q[a] >= m.n[a] ? 1 : 0);
                out2 |= e[a] != 0;
            }
            if (out2) {
                c.blk = g.nbr[nbr_dir(m, e)];
#pragma unroll
                for (int a = 0; a < 3; ++a) q[a] -= e[a] * m.n[a];
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) p[a] = q[a];
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) c.p[a] = p[a];
    return c;
}

// The boundary functor of a cell's source, on its primitives.
template <class FT, int NV>
__device__ __forceinline__ void cell_functor(const MeshView<FT> &m, const CellSrc &c, FT *w) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (c.flip == a) {
            w[MOM + a] = w[MOM + a] * -1;
            if constexpr (NV == 8) {
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    if (k != a) w[BCC + k] = -w[BCC + k];
            }
        }
        if (c.clamp >= 0 && (c.clamp >> 1) == a) {
            const int side = c.clamp & 1;
            if (w[MOM + a] * (side ? -1 : 1) > 0) w[MOM + a] = 0;
        }
    }
    if (c.fixd) {             // hydro / mhd phys_functors.h fixed_t
#pragma unroll
        for (int v = 0; v < 5; ++v) w[v] = (FT)m.fix_w[v];
        if constexpr (NV == 8) {
#pragma unroll
            for (int k = 0; k < 3; ++k) w[BCC + k] = (FT)m.fix_b[k];
        }
    }
}

// Load the primitive vector of cell pin of block b.
template <class FT, int NV>
__device__ __forceinline__ void load_cell(const MeshView<FT> &m, int b, const int *pin, FT *w) {
    const CellSrc c = cell_src<FT, NV>(m, b, pin);
    const FT *src = m.W + (size_t)c.blk * NV * m.ncell + cidx(m.n, c.p[0], c.p[1], c.p[2]);
#pragma unroll
    for (int v = 0; v < NV; ++v) w[v] = src[(size_t)v * m.ncell];
    cell_functor<FT, NV>(m, c, w);
}

// Normal face field of block b at face p (component c); transverse indices
// may sit one row outside the block (MHD transverse ghost lines), which the
// reference fills by the tangential face-field exchange
// (mhd/boundary/comm_functions.h:433-465).
template <class FT>
__device__ __forceinline__ double load_bf(const MeshView<FT> &m, int b, int slot, int c,
                                          const int *pin) {
    int p[3] = {pin[0], pin[1], pin[2]};
    int d[3] = {0, 0, 0};
    bool out = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (a == c) continue;
        d[a] = p[a] < 0 ? -1 : (p[a] >= m.n[a] ? 1 : 0);
        out |= d[a] != 0;
    }
    int blk = b;
    if (out) {
        const BlockGeo &g = m.geo[b];
        if (g.xface) {
            // mhd/integrator/data.h:108-140: a transverse ghost line next to a
            // cross-level face takes the normal field from the cell value of w
            int bit = 0;
#pragma unroll
            for (int a = 0; a < 3; ++a)
                if (d[a]) bit = 1 << (2 * a + (d[a] > 0));
            if (g.xface & bit) {
                FT w[8];
                load_cell<FT, 8>(m, b, pin, w);
                return (double)w[BCC + c];
            }
        }
        blk = g.nbr[nbr_dir(m, d)];
        if (blk < 0) {
            // physical side (mhd/boundary/phys.h:178-229, phys_functors.h
            // :10-137): the tangential face field of the ghost cell next to
            // the side; free / outflow copy the boundary cell's, reflect
            // takes minus the one at -i (two cells in).  Along the
            // component's own axis the source row is clamped into the block
            // where that axis is physical at the top.
            int a = 0;
#pragma unroll
            for (int x = 0; x < 3; ++x)
                if (d[x]) a = x;
            const int side = d[a] > 0;
            const int kind = m.bnd[2 * a + side];
            if (kind == 4) return m.fix_b[c];
            double sgn = 1;
            if (kind == 3) {
                p[a] = side ? m.n[a] - 2 : 1;
                sgn = -1;
            } else {
                p[a] = side ? m.n[a] - 1 : 0;
            }
            if (((g.phy >> (2 * c + 1)) & 1) && p[c] >= m.n[c]) p[c] = m.n[c] - 1;
            return sgn * m.BF[(((size_t)b * 2 + slot) * 3 + c) * m.nface + fidx(m.n, p[0], p[1], p[2])];
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) p[a] -= d[a] * m.n[a];
    }
    return m.BF[(((size_t)blk * 2 + slot) * 3 + c) * m.nface + fidx(m.n, p[0], p[1], p[2])];
}

// Wave64 + workgroup min reduction of a double; lane 0 of the workgroup
// returns the result.
__device__ __forceinline__ double block_min(double v) {
    __shared__ double red[kThreads / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = pmin(v, __shfl_xor(v, off, 64));
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) red[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < (int)(blockDim.x >> 6); ++i) v = pmin(v, red[i]);
    }
    return v;
}

// ------------------------------------------------------------------- c2p
// Primitives of cell (i, j, k) of block b (hydro/eos/adiabatic.h:211-259,
// mhd/eos/adiabatic.h:127-235) from its conserved state in slot `slot`, which
// the caller has loaded into cons: healed values in cons, prim, for MHD the
// cell-centred B from the face average and the squares and face maxima that
// the CFL speeds use.  heal_rho: rho was raised to its floor; moved: the energy
// that the slot should hold differs from what it holds (the subtract / add
// round trip of the magnetic part, or a healed pressure).  Returns c_s^2.
template <class FT, bool MHD>
__device__ __forceinline__ double cell_c2p(const MeshView<FT> &m, int b, int slot, int i, int j, int k,
                                           double *cons, double *prim, double *bc, double *bc_2,
                                           double *b_max, bool &heal_rho, bool &moved) {
    const EosPar e{m.gamma, m.cfl, m.d_floor, m.t_floor};
    if constexpr (MHD) {
        const double *BF = m.BF + ((size_t)b * 2 + slot) * 3 * m.nface;
        double e_m(0);
        const size_t f0 = fidx(m.n, i, j, k);
        const size_t sh[3] = {1, (size_t)(m.n[0] + 1), (size_t)(m.n[0] + 1) * (m.n[1] + 1)};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            // a thin (one-cell) axis has one face per cell, both sides
            // of it (mhd/eos/adiabatic.h:164-177)
            const double b_l = BF[(size_t)a * m.nface + f0];
            const double b_r = m.n[a] < 2 ? b_l : BF[(size_t)a * m.nface + f0 + sh[a]];
            const double bc_m = (b_l + b_r) / 2;
            bc[a] = bc_m;
            const double bcs2 = bc_m * bc_m;
            e_m += bcs2;
            bc_2[a] = bcs2;
            b_max[a] = pmax(kfabs(b_l), kfabs(b_r));
        }
        e_m /= 2;
        const double e_in = cons[ENE];
        bool he;
        cons[ENE] -= e_m;
        const double cs2 = c2p(cons, prim, e, heal_rho, he);
        cons[ENE] += e_m;
        moved = cons[ENE] != e_in;
        return cs2;
    } else {
        return c2p(cons, prim, e, heal_rho, moved);
    }
}

// Global CFL reduction and the dt / t bookkeeping of redc_dt_start/finish
// (mesh/cycle/cycle.cpp:77-115): p_dt = min(p_dt, CFL), dt_use clamped to
// t_lim when topping up, t advanced, next seed = dt_use * dt_expand.
__device__ __forceinline__ void take_dt(TimeState *ts, double cfl_dt) {
    const double p = __builtin_fmin(cfl_dt, ts->p_dt);
    const double dt_use = ts->top_up ? (p < ts->t_lim - ts->t ? p : ts->t_lim - ts->t) : p;
    if (ts->top_up) {
        const double tn = dt_use + ts->t;
        ts->t = tn < ts->t_lim ? tn : ts->t_lim;
    } else {
        ts->t = dt_use + ts->t;
    }
    ts->dt_use = dt_use;
    ts->p_dt = dt_use * ts->dt_expand;
}

// c2p of one substep: primitives with floors written back to the conserved
// slot, and at substep 0 the per-cell CFL dt reduced per workgroup.
//
// FIN (substep 0 of small meshes): the workgroup that finishes last in its
// time group also takes the group's dt, and the stop rule of cycle::step
// (mesh/cycle/cycle.cpp:143-144) is evaluated here, so that no launch is
// spent on either (k_cycle_begin and k_dt_finalize, together 6 to 9 us of a
// cycle; on large meshes the arrivals would cost more than the launches).
// arrived[g] counts the group's workgroups and is left at 0.
constexpr int kFinWaves = 16;          // waves of k_dt_finalize
template <class FT, bool MHD, bool FIN>
__global__ void __launch_bounds__(kThreads) k_c2p(MeshView<FT> m, int step, const int *grp_first,
                                                  int *arrived) {
    const int b = blockIdx.y, grp = m.geo[b].grp;
    TimeState *ts = m.ts + grp;
    const bool skip = FIN ? ts->t >= ts->t_lim : ts->skip != 0;
    if (!FIN && skip) return;
    constexpr int NV = MHD ? 8 : 5;
    const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    double dtc = (double)FLT_MAX;
    if (c < m.ncell && !skip) {
        // loaded before the 64-bit divisions that give i, j, k, which hydro does
        // not need (128^3 MHD, a launch: with the loads after them 47.2 us mixed
        // and 56.4 FP64, so 44.6 and 54.8; 256^3 hydro mixed with and without
        // the divisions 180 and 171)
        double *U = m.U + ((size_t)b * 2 + step) * 5 * m.ncell + c;
        double cons[5], prim[5], bc[3], bc_2[3], b_max[3];
#pragma unroll
        for (int v = 0; v < 5; ++v) cons[v] = U[(size_t)v * m.ncell];
        const int i = (int)(c % m.n[0]);
        const int j = (int)((c / m.n[0]) % m.n[1]);
        const int k = (int)(c / ((size_t)m.n[0] * m.n[1]));
        bool heal_rho, moved;
        const double cs2 = cell_c2p<FT, MHD>(m, b, step, i, j, k, cons, prim, bc, bc_2, b_max, heal_rho, moved);
        const BlockGeo &g = m.geo[b];
        FT *W = m.W + (size_t)b * NV * m.ncell + c;
        // the slot is written only where it does not hold the value already
        if (moved) U[(size_t)ENE * m.ncell] = cons[ENE];
        if (heal_rho) U[0] = cons[RHO];
#pragma unroll
        for (int v = 0; v < 5; ++v) W[(size_t)v * m.ncell] = (FT)prim[v];
        if constexpr (MHD) {
#pragma unroll
            for (int a = 0; a < 3; ++a) W[(size_t)(BCC + a) * m.ncell] = (FT)bc[a];
            if (m.EC) {     // mhd/eos/adiabatic.h:214-219, from the stored values
                const FT B[3] = {(FT)bc[0], (FT)bc[1], (FT)bc[2]};
                const FT V[3] = {(FT)prim[MOM], (FT)prim[MOM + 1], (FT)prim[MOM + 2]};
                FT *E = m.EC + (size_t)b * 3 * m.ncell + c;
                E[0] = B[1] * V[2] - B[2] * V[1];
                E[m.ncell] = B[2] * V[0] - B[0] * V[2];
                E[2 * m.ncell] = B[0] * V[1] - B[1] * V[0];
            }
            if (step == 0)
                dtc = std::is_same_v<FT, float>
                          ? dt_mhd_mixed(prim, bc_2, b_max, g.dx, m.ndim, m.gamma, m.cfl)
                          : dt_mhd(prim, bc_2, b_max, g.dx, m.ndim, m.gamma, m.cfl);
        } else if (step == 0) {
            dtc = dt_hydro(prim, cs2, g.dx, m.ndim, m.cfl);
        }
    }
    if constexpr (!FIN) {
        if (step == 0) {
            const double r = block_min(dtc);
            if (threadIdx.x == 0) m.dt_part[(size_t)b * gridDim.x + blockIdx.x] = r;
        }
    } else {
        const double r = block_min(dtc);
        const int first = grp_first[grp], last = grp_first[grp + 1];
        __shared__ bool s_last;
        if (threadIdx.x == 0) {
            __hip_atomic_store(m.dt_part + (size_t)b * gridDim.x + blockIdx.x, r, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            const int n = __hip_atomic_fetch_add(arrived + grp, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
            s_last = n + 1 == (last - first) * (int)gridDim.x;
        }
        __syncthreads();
        if (!s_last) return;
        // the partials in k_dt_finalize's order, 64 of them a wave's: pmin keeps
        // or drops a NaN by its place, and a state that holds one is to take the
        // same dt on either side of the line
        __shared__ double s_min[kFinWaves];
        const double *part = m.dt_part + (size_t)first * gridDim.x;
        const int n = (last - first) * (int)gridDim.x, waves = (n + 63) / 64;
        for (int w = threadIdx.x >> 6; w < waves; w += kThreads / 64) {
            const int i = w * 64 + (threadIdx.x & 63);
            double v = (double)FLT_MAX;
            if (i < n) v = pmin(v, __hip_atomic_load(part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v = pmin(v, __shfl_xor(v, off, 64));
            if ((threadIdx.x & 63) == 0) s_min[w] = v;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double v = s_min[0];
            for (int w = 1; w < waves; ++w) v = pmin(v, s_min[w]);
            if (waves < kFinWaves) v = pmin(v, (double)FLT_MAX);     // its idle waves
            ts->skip = skip ? 1 : 0;
            if (!skip) {
                ts->cycles += 1;
                take_dt(ts, v);
            }
            __hip_atomic_store(arrived + grp, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// ------------------------------------------------------------------ flux
// One thread per face of the sweep along `axis` (PLM + HLLC / HLLD), the
// flux_kernel of prototypes/integrator.h:14-32 with hydro/integrator/data.h
// :334-352 (hydro) or mhd/integrator/data.h:53-141 (MHD lines, including the
// transverse ghost lines) for the pencil, PLM per face
// (hydro/reconstruct/plm.h:116-153, mhd/reconstruct/plm.h:18-50).
//
// FP64 takes the functions of kr_exact64.h.  Fewer instructions helped little
// here: the three sweeps over 442 MHD blocks of 8^3 went from 36.6, 36.4 and
// 34.9 us to 35.2, 34.8 and 32.3 (seven waves a SIMD, of which 148 registers
// let three run at a time).
template <class FT, bool MHD, int AXIS>
__global__ void __launch_bounds__(kThreads) k_flux(MeshView<FT> m, int step) {
    constexpr int axis = AXIS;
    if (m.ts[m.geo[row_block(m)].grp].skip) return;
    constexpr int NV = MHD ? 8 : 5;
    const int b = row_block(m);
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= m.nfa[axis]) return;
    int D[3], o[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        D[a] = m.n[a] + (a == axis ? 1 : 2);
        o[a] = a == axis ? 0 : 1;
    }
    int p[3];
    p[0] = (int)(t % D[0]) - o[0];
    p[1] = (int)((t / D[0]) % D[1]) - o[1];
    p[2] = (int)(t / ((size_t)D[0] * D[1])) - o[2];
    constexpr int a1 = (axis + 1) % 3, a2 = (axis + 2) % 3;
    const bool in1 = p[a1] >= 0 && p[a1] < m.n[a1];
    const bool in2 = p[a2] >= 0 && p[a2] < m.n[a2];
    if constexpr (MHD) {
        // transverse ghost lines exist only along active axes
        // (mhd/integrator/integrator.h:152-155)
        if (!in1 && !in2) return;
        if ((!in1 && m.n[a1] < 2) || (!in2 && m.n[a2] < 2)) return;
    } else {
        if (!in1 || !in2) return;
    }
    FT q[4][NV];
    const int f = p[axis];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        int pc[3] = {p[0], p[1], p[2]};
        pc[axis] = f - 2 + s;
        load_cell<FT, NV>(m, b, pc, q[s]);
    }
    FT ql[NV], qr[NV], flx[NV];
    if constexpr (std::is_same_v<FT, float>) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            if (MHD && v == BCC + axis) continue;
            plm_fast(q[0][v], q[1][v], q[2][v], q[3][v], ql[v], qr[v]);
        }
    } else {
        FT lo[2 * NV], hi[2 * NV], t[2 * NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const bool bn = MHD && v == BCC + axis;      // taken from the face below
            lo[v] = bn ? 0 : q[1][v] - q[0][v];
            hi[v] = lo[NV + v] = bn ? 0 : q[2][v] - q[1][v];
            hi[NV + v] = bn ? 0 : q[3][v] - q[2][v];
        }
        plm_inc64<2 * NV>(lo, hi, t);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            ql[v] = q[1][v] + t[v];
            qr[v] = q[2][v] - t[NV + v];
        }
    }
    if constexpr (MHD) {
        const FT bn = (FT)load_bf(m, b, step, axis, p);
        ql[BCC + axis] = bn;
        qr[BCC + axis] = bn;
    }
    face_flux<FT, MHD, AXIS>(ql, qr, flx, Gam64{m.gamma, m.cv, m.ge});
    FT *F = m.F[axis] + (size_t)b * NV * m.nfa[axis] + t;
#pragma unroll
    for (int v = 0; v < NV; ++v) F[(size_t)v * m.nfa[axis]] = flx[v];
}

// ------------------------------------------------------------------- EMF
// Edge EMF of an edge between two active axes (k_emf's expressions, with its
// rounding also in FP32): cell E at the four corners and the face EMFs and
// mass fluxes of both directions.
template <class FT>
__device__ __forceinline__ FT corner_emf(FT ec11, FT ec10, FT ec00, FT ec01, FT efm1, FT efp1, FT rp1,
                                         FT rm1, FT efm2, FT efp2, FT rp2, FT rm2) {
    const FT w_e = (FT)0.25f;
    FT ee = 0;
    ee += w_e * (efm1 + efp1);
    {
        const FT de_p = (rp1 > 0 ? (ec01 - efm1) : (ec11 - efp1));
        const FT de_m = (rm1 > 0 ? -(ec00 - efm1) : -(ec10 - efp1));
        ee += w_e * (de_m - de_p);
    }
    ee += w_e * (efm2 + efp2);
    {
        const FT de_p = (rp2 > 0 ? (ec10 - efm2) : (ec11 - efp2));
        const FT de_m = (rm2 > 0 ? -(ec00 - efm2) : -(ec01 - efp2));
        ee += w_e * (de_m - de_p);
    }
    return ee;
}

template <class FT>
__device__ __forceinline__ FT ec_at(const MeshView<FT> &m, int b, const int *p, const int *ax) {
    bool in = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) in &= p[a] >= 0 && p[a] < m.n[a];
    if (in)     // the block's own cell: the c2p value (equal to B x v of its w)
        return m.EC[((size_t)b * 3 + ax[0]) * m.ncell + cidx(m.n, p[0], p[1], p[2])];
    FT w[8];
    load_cell<FT, 8>(m, b, p, w);
    return w[BCC + ax[1]] * w[MOM + ax[2]] - w[BCC + ax[2]] * w[MOM + ax[1]];
}

template <class FT>
__device__ __forceinline__ FT flux_at(const MeshView<FT> &m, int b, int a, const int *p, int v) {
    return m.F[a][((size_t)b * 8 + v) * m.nfa[a] + xidx(m.n, a, p)];
}

// Edge EMF with the corner-upwind correction, mhd/integrator/integrator.h
// :189-327.  Cell-centred E outside the block is B x v from the neighbour's
// primitives (:201-213); inside it equals the c2p ec.  Thin (one-cell) axes
// come last (m.ndim counts the active ones): they carry one edge layer, no
// shift, no flux and no corner upwinding, and an edge next to one takes the
// surviving sweep at weight 0.5 (:221-300).
template <class FT, int AX>
__device__ __forceinline__ FT edge_at(const MeshView<FT> &m, int b, int *i) {
    constexpr int ax = AX, ax_1 = (AX + 1) % 3, ax_2 = (AX + 2) % 3;
    const int n_dm = m.ndim;
    const bool th_1 = ax_1 >= n_dm, th_2 = ax_2 >= n_dm;
    const int axis[3] = {ax, ax_1, ax_2};
    FT ec[2][2];
    ec[1][1] = ec_at(m, b, i, axis);
    if (!th_1) --i[ax_1];
    ec[1][0] = ec_at(m, b, i, axis);
    if (!th_2) --i[ax_2];
    ec[0][0] = ec_at(m, b, i, axis);
    if (!th_1) ++i[ax_1];
    ec[0][1] = ec_at(m, b, i, axis);
    if (!th_2) ++i[ax_2];
    FT ee = 0;
    const FT w_e = (th_1 || th_2) ? (FT)0.5f : (FT)0.25f;
#pragma unroll
    for (int pi = 0; pi < 2; ++pi) {
        const int a_para = pi == 0 ? ax_1 : ax_2;
        const int a_perp = pi == 0 ? ax_2 : ax_1;
        const bool thn_p = a_perp >= n_dm;
        if (a_para < n_dm) {
            if (!thn_p) --i[a_perp];
            const FT ef_m = flux_at(m, b, a_para, i, BCC + ax);
            if (!thn_p) ++i[a_perp];
            const FT ef_p = flux_at(m, b, a_para, i, BCC + ax);
            ee += w_e * (ef_m + ef_p);
            if (!thn_p) {
                const FT frho_p = flux_at(m, b, a_perp, i, RHO);
                --i[a_para];
                const FT frho_m = flux_at(m, b, a_perp, i, RHO);
                ++i[a_para];
                const FT de_p = (frho_p > 0 ? (ec[0][1] - ef_m) : (ec[1][1] - ef_p));
                const FT de_m = (frho_m > 0 ? -(ec[0][0] - ef_m) : -(ec[1][0] - ef_p));
                ee += w_e * (de_m - de_p);
            }
        }
        if (pi == 0) {
            const FT swp = ec[0][1];
            ec[0][1] = ec[1][0];
            ec[1][0] = swp;
        }
    }
    return ee;
}

// One grid layer (z) per edge direction: an edge waits for its cells, then
// for its fluxes, behind the branches that find them, and a thread that took
// its three edges one after another did so three times in a row (442 FP64
// blocks of 8^3: 38.2 us, with layers 28.3; a cycle of the staged mixed form
// at 32^3 122.5 and 104.0 us, at 128^3 1,010 and 953).
template <class FT>
__global__ void __launch_bounds__(kThreads) k_emf(MeshView<FT> m) {
    if (m.ts[m.geo[row_block(m)].grp].skip) return;
    const int b = row_block(m), ax = blockIdx.z;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= m.nface) return;
    int i[3];
    i[0] = (int)(t % (m.n[0] + 1));
    i[1] = (int)((t / (m.n[0] + 1)) % (m.n[1] + 1));
    i[2] = (int)(t / ((size_t)(m.n[0] + 1) * (m.n[1] + 1)));
    for (int a = m.ndim; a < 3; ++a)
        if (i[a] > 0) return;
    FT *EE = m.EE + ((size_t)b * 3 + ax) * m.nface + t;
    if (ax == 0 && i[0] < m.n[0]) *EE = edge_at<FT, 0>(m, b, i);
    if (ax == 1 && i[1] < m.n[1]) *EE = edge_at<FT, 1>(m, b, i);
    if (ax == 2 && i[2] < m.n[2]) *EE = edge_at<FT, 2>(m, b, i);
    // boundary-plane advective edge EMF of a high out / fre side
    // (mhd/integrator/integrator.h:328-381): the interior cell's value with
    // v = w[mom] / rho as written there; later axes overwrite earlier ones
    const BlockGeo &g = m.geo[b];
    if (g.phy)
        for (int a = 0; a < 3; ++a) {
            if (a == ax || i[a] != m.n[a] || m.n[a] < 2 || !((g.phy >> (2 * a + 1)) & 1)) continue;
            const int k = m.bnd[2 * a + 1];
            if (k != 1 && k != 2) continue;
            int jc[3] = {i[0], i[1], i[2]};
            --jc[a];
            FT w[8];
            load_cell<FT, 8>(m, b, jc, w);
            const FT irho = (FT)1 / pmax(w[RHO], (FT)1e-30);
            FT v_c[3], b_c[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                v_c[q] = w[MOM + q] * irho;
                b_c[q] = w[BCC + q];
            }
            const int a1 = mod3(a + 1), a2 = mod3(a + 2);
            *EE = ax == a1 ? v_c[a] * b_c[a2] - v_c[a2] * b_c[a] : v_c[a1] * b_c[a] - v_c[a] * b_c[a1];
        }
}

// ---------------------------------------------------------------- update
// Flux divergence + Heun slot (hydro/integrator/integrator.h:56-68, 156-182,
// 241-265; rk2.h:20-41) and, for MHD, the CT update of the face field
// (mhd/integrator/integrator.h:385-462 with rk2.h:191-205).
//
// One point of the update: the cell at face-box point t of block b (when
// it is a cell) and, for MHD, the faces of that point.  edge(EE, c, idx,
// i, s) reads the edge EMF of component c at edge-box index idx, EE being
// block b's edges; the edge sits at the point's coordinates i, one further
// along axis s when s >= 0.  finish(i, uu) may add to the cell's new state
// before it is stored.
template <class FT, bool MHD, class EdgeRead, class CellFinish>
__device__ __forceinline__ void update_point(const MeshView<FT> &m, int b, size_t t, int step,
                                             EdgeRead edge, CellFinish finish) {
    constexpr int NV = MHD ? 8 : 5;
    int i[3];
    const int e0 = m.n[0] + (MHD ? 1 : 0), e1 = m.n[1] + (MHD ? 1 : 0);
    i[0] = (int)(t % e0);
    i[1] = (int)((t / e0) % e1);
    i[2] = (int)(t / ((size_t)e0 * e1));
    const double dt = m.ts[m.geo[b].grp].dt_use * (step == 0 ? 1.0 : 0.5);
    const BlockGeo &g = m.geo[b];
    // grid layer: -1 all of the point, else 0 its cell, 1 + a its face along a
    const int part = MHD && gridDim.z > 1 ? (int)blockIdx.z : -1;
    if (part <= 0 && i[0] < m.n[0] && i[1] < m.n[1] && i[2] < m.n[2]) {
        const size_t c = cidx(m.n, i[0], i[1], i[2]);
        const double *Us = m.U + ((size_t)b * 2 + step) * 5 * m.ncell + c;
        double *Ut = m.U + ((size_t)b * 2 + (1 - step)) * 5 * m.ncell + c;
        double uu[5];
        if (step == 0) {
#pragma unroll
            for (int v = 0; v < 5; ++v) uu[v] = Us[(size_t)v * m.ncell];
        } else {
#pragma unroll
            for (int v = 0; v < 5; ++v)
                uu[v] = (Us[(size_t)v * m.ncell] + Ut[(size_t)v * m.ncell]) * 0.5f;
        }
        const double dt_dv = dt / g.vol;
        // All face fluxes are loaded before the first is used, also those of
        // faces that the sums below leave out (they lie in the flux box): a
        // cell waits for memory once and not once behind each condition
        // (k_smr_update, mixed, 442 blocks of 16^3: 142 -> 113 us).
        FT f0[3][5], f1[3][5];
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            if (ax >= m.ndim) continue;
            int p1[3] = {i[0], i[1], i[2]};
            ++p1[ax];
            const size_t x0 = xidx(m.n, ax, i), x1 = xidx(m.n, ax, p1);
            const FT *F = m.F[ax] + (size_t)b * NV * m.nfa[ax];
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                f0[ax][v] = F[(size_t)v * m.nfa[ax] + x0];
                f1[ax][v] = F[(size_t)v * m.nfa[ax] + x1];
            }
        }
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            if (ax >= m.ndim) continue;
            // faces whose neighbour is finer are skipped here and added with
            // the restricted flux afterwards (integrator.h:156-182 null_l/r)
            const bool n0 = ((g.rface >> (2 * ax)) & 1) && i[ax] == 0;
            const bool n1 = ((g.rface >> (2 * ax + 1)) & 1) && i[ax] + 1 == m.n[ax];
            const FT fa = (FT)(g.sfc[ax] * dt_dv);
            const bool u0 = !n0 && fa > 0, u1 = !n1 && fa > 0;
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                double res(0);
                res = u0 ? res + (double)(fa * f0[ax][v]) : res;
                res = u1 ? res - (double)(fa * f1[ax][v]) : res;
                uu[v] += res;
            }
        }
        finish(i, uu);
#pragma unroll
        for (int v = 0; v < 5; ++v) Ut[(size_t)v * m.ncell] = uu[v];
    }
    if constexpr (MHD) {
        // the index-1 slot of a thin axis is not a face of the block: it
        // is never computed, and every reader takes slot 0 for both sides
        for (int a = m.ndim; a < 3; ++a)
            if (i[a] > 0) return;
        const FT *EE = m.EE + (size_t)b * 3 * m.nface;
        double *Bs = m.BF + ((size_t)b * 2 + step) * 3 * m.nface + t;
        double *Bt = m.BF + ((size_t)b * 2 + (1 - step)) * 3 * m.nface + t;
        const size_t sh[3] = {1, (size_t)(m.n[0] + 1), (size_t)(m.n[0] + 1) * (m.n[1] + 1)};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int ax_1 = mod3(a + 1), ax_2 = mod3(a + 2);
            if ((part >= 0 && part != a + 1) || i[ax_1] >= m.n[ax_1] || i[ax_2] >= m.n[ax_2]) continue;
            // an edge pair spanning a thin axis vanishes
            // (mhd/integrator/integrator.h:419-447)
            const bool th_1 = ax_1 >= m.ndim, th_2 = ax_2 >= m.ndim;
            // FP64 edge circulation (also in the mixed form: the EMF is
            // widened before the product so CT keeps div B at round-off).
            double db = th_2 ? 0.0 : (double)edge(EE, ax_1, t, i, -1) * g.dx[ax_1];
            if (!th_1) {
                db -= (double)edge(EE, ax_2, t, i, -1) * g.dx[ax_2];
                db += (double)edge(EE, ax_2, t + sh[ax_1], i, ax_1) * g.dx[ax_2];
            }
            if (!th_2) db -= (double)edge(EE, ax_1, t + sh[ax_2], i, ax_2) * g.dx[ax_1];
            // the thin face family's area (sfc_thin, integrator.h:74-81)
            const double sfc = a >= m.ndim ? g.dx[ax_1] * g.dx[ax_2] : g.sfc[a];
            db *= (sfc > 0 ? (double)(-dt / sfc) : (double)(0));
            const double bs = Bs[(size_t)a * m.nface];
            Bt[(size_t)a * m.nface] =
                db + (step == 0 ? bs : (bs + Bt[(size_t)a * m.nface]) / 2);
        }
    }
}

template <class FT, bool MHD>
__global__ void __launch_bounds__(kThreads) k_update(MeshView<FT> m, int step) {
    if (m.ts[m.geo[row_block(m)].grp].skip) return;
    const int b = row_block(m);
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (MHD ? m.nface : m.ncell)) return;
    update_point<FT, MHD>(
        m, b, t, step,
        [&](const FT *EE, int c, size_t idx, const int *, int) -> FT {
            return EE[(size_t)c * m.nface + idx];
        },
        [](const int *, double *) {});
}

// Max |div B| per workgroup (diagnostic): sum over axes of the face
// difference divided by the cell width, slot 0.
template <class FT>
__global__ void __launch_bounds__(kThreads) k_divb(MeshView<FT> m, double *part) {
    const int b = blockIdx.y;
    const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0;
    if (c < m.ncell) {
        const int i = (int)(c % m.n[0]);
        const int j = (int)((c / m.n[0]) % m.n[1]);
        const int k = (int)(c / ((size_t)m.n[0] * m.n[1]));
        const double *BF = m.BF + (size_t)b * 2 * 3 * m.nface;
        const size_t f0 = fidx(m.n, i, j, k);
        const size_t sh[3] = {1, (size_t)(m.n[0] + 1), (size_t)(m.n[0] + 1) * (m.n[1] + 1)};
        double s = 0;
        for (int a = 0; a < m.ndim; ++a)      // no variation along a thin axis
            s += (BF[(size_t)a * m.nface + f0 + sh[a]] - BF[(size_t)a * m.nface + f0]) / m.geo[b].dx[a];
        v = kfabs(s);
    }
    v = -v;
    const double r = block_min(v);
    if (threadIdx.x == 0) part[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = -r;
}

}  // namespace kr
