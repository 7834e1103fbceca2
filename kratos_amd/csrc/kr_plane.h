// kr_plane.h -- the whole stage of a 2-D or 1-D mesh in one launch: face
// fluxes, edge EMFs, the Heun update and constrained transport, and at
// substep 1 also the primitives.
//
// Thin meshes are small (256^2 cells are 1,024 tiles), so what bounds them
// is the number of dependent launches of a cycle, each 5 to 17 us of which
// little is work: the staged kernels take twelve.  One workgroup here owns a
// TX x TY tile (TY = 1: a 1-D mesh): it loads the primitives of the tile and a 2-cell halo into
// LDS, solves the tile's x and y faces (for MHD with the ghost lines that the
// corner-upwind EMFs read), forms the edge EMFs in LDS and updates its own
// cells and faces.  With k_c2p's FIN form before substep 0 a cycle is three
// launches.
//
// C2P (substep 1): the primitives of the tile and its halo come straight
// from slot 1, by k_c2p's arithmetic, instead of from W; a neighbour's healed
// values are not needed, and the owned cells' are kept in LDS for the update
// (nothing reads slot 1 after it).  Substep 0 cannot do so: the healed slot 0
// is read again by substep 1.  Each substep reads only what the launch
// before it wrote (slot `step`, W) and its own cells of the slot it writes.
//
// The arithmetic is that of the staged kernels (k_flux, k_emf, k_update), in
// their order: both forms give their state bit for bit (FP64 through
// kr_exact64.h).  Tiles may overhang the block: any block size.
#pragma once

#include "kr_exact64.h"
#include "kr_staged.h"

namespace kr {

template <class FT, bool MHD, int TX, int TY, int NT, bool C2P>
__global__ void __launch_bounds__(NT) k_plane(MeshView<FT> m, int step) {
    constexpr int NV = MHD ? 8 : 5;
    constexpr bool two = TY > 1;                         // y is active
    constexpr int G = MHD && two ? 1 : 0;                // ghost lines of the faces
    constexpr int HX = TX + 4, HY = two ? TY + 4 : 1, NCOL = HX * HY, NOWN = TX * TY;
    constexpr int NFX = (TX + 1) * (TY + 2 * G), NFY = two ? (TX + 2 * G) * (TY + 1) : 0, NF = NFX + NFY;
    constexpr int NP = two ? (TX + 1) * (TY + 1) : TX + 1;   // points: cells and high faces
    static_assert(NCOL <= NT, "one cell of tile and halo per thread");
    static_assert(NF <= NT, "one face per thread");
    static_assert(NP <= NT, "one point per thread");
    if (m.ts[m.geo[blockIdx.y].grp].skip) return;
    const int tid = threadIdx.x;
    const int b = blockIdx.y;
    const int ntx = (m.n[0] + TX - 1) / TX;
    const int x0 = (blockIdx.x % ntx) * TX, y0 = (blockIdx.x / ntx) * TY;
    const int n0 = m.n[0], n1 = m.n[1];
    const size_t nc = m.ncell;
    const BlockGeo &g = m.geo[b];
    const double dt = m.ts[g.grp].dt_use * (step == 0 ? 1.0 : 0.5);

    __shared__ FT sW[NV][NCOL];
    __shared__ FT sF[5][NF];            // face fluxes, mesh frame
    __shared__ FT sE[MHD ? 2 : 1][NF];  // face EMFs: E_y of x faces / E_x of y faces, and E_z
    __shared__ FT sEd[MHD ? 3 : 1][NP]; // edge EMFs
    __shared__ double sU[C2P ? 2 : 1][NOWN];   // healed rho and E of the owned cells
    auto col = [](int x, int y) { return (two ? y + 2 : 0) * HX + (x + 2); };
    auto fxi = [](int x, int y) { return (y + G) * (TX + 1) + x; };
    auto fyi = [](int x, int y) { return NFX + y * (TX + 2 * G) + (x + G); };
    auto edi = [](int x, int y) { return y * (TX + 1) + x; };

    // ---------------------------------------------- primitives of the tile
    if (tid < NCOL) {
        const int x = tid % HX - 2, y = two ? tid / HX - 2 : 0;
        const int gx = x0 + x, gy = y0 + y;
        const bool ox = gx < -G || gx >= n0 + G, oy = gy < -G || gy >= n1 + G;
        // the corners of the halo enter no flux; a thin axis has no halo, and
        // hydro reads ghosts along one axis only
        const bool need = gx <= n0 + 1 && gy <= n1 + 1 &&
                          ((x >= -G && x < TX + G) || (y >= -G && y < TY + G)) && !(ox && oy);
        if (need) {
            const int p[3] = {gx, gy, 0};
            FT w[NV];
            if constexpr (C2P) {
                const CellSrc c = cell_src<FT, NV>(m, b, p);
                double cons[5], prim[5], bc[3], bc_2[3], b_max[3];
                bool heal_rho, moved;
                const double *U = m.U + ((size_t)c.blk * 2 + step) * 5 * nc + cidx(m.n, c.p[0], c.p[1], c.p[2]);
#pragma unroll
                for (int v = 0; v < 5; ++v) cons[v] = U[(size_t)v * nc];
                cell_c2p<FT, MHD>(m, c.blk, step, c.p[0], c.p[1], c.p[2], cons, prim, bc, bc_2, b_max,
                                  heal_rho, moved);
#pragma unroll
                for (int v = 0; v < 5; ++v) w[v] = (FT)prim[v];
                if constexpr (MHD) {
#pragma unroll
                    for (int a = 0; a < 3; ++a) w[BCC + a] = (FT)bc[a];
                }
                cell_functor<FT, NV>(m, c, w);
                if (x >= 0 && x < TX && y >= 0 && y < TY) {
                    sU[0][y * TX + x] = cons[RHO];
                    sU[1][y * TX + x] = cons[ENE];
                }
            } else {
                load_cell<FT, NV>(m, b, p, w);
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) sW[v][tid] = w[v];
        }
    }
    __syncthreads();

    // ---------------------------------------------- face fluxes
    if (tid < NF) {
        const bool xf = tid < NFX;
        int x, y;
        if (xf || !two) {
            x = tid % (TX + 1);
            y = tid / (TX + 1) - G;
        } else {
            x = (tid - NFX) % (TX + 2 * G) - G;
            y = (tid - NFX) / (TX + 2 * G);
        }
        const int gx = x0 + x, gy = y0 + y;
        const bool need = xf ? gx <= n0 && gy < n1 + G : gy <= n1 && gx < n0 + G;
        if (need) {
            const int a = xf ? 0 : 1, st = xf ? 1 : HX;
            const int c = col(x, y);
            FT ql[NV], qr[NV], flx[NV];
            // rotated frame: slot k holds mesh variable perm(k)
            auto perm = [&](int k) {
                if (k < MOM) return k;
                const int o = k < BCC ? MOM : BCC;
                const int r = a + k - o;
                return o + (r >= 3 ? r - 3 : r);
            };
            if constexpr (std::is_same_v<FT, float>) {
#pragma unroll
                for (int k = 0; k < NV; ++k) {
                    if (MHD && k == BCC) continue;
                    const FT *q = &sW[perm(k)][c];
                    plm_fast(q[-2 * st], q[-st], q[0], q[st], ql[k], qr[k]);
                }
            } else {
                constexpr int N = MHD ? 7 : 5;
                FT lo[2 * N], hi[2 * N], t[2 * N];
#pragma unroll
                for (int k = 0, j = 0; k < NV; ++k) {
                    if (MHD && k == BCC) continue;
                    const FT *q = &sW[perm(k)][c];
                    ql[k] = q[-st];
                    qr[k] = q[0];
                    lo[j] = ql[k] - q[-2 * st];
                    hi[j] = lo[N + j] = qr[k] - ql[k];
                    hi[N + j] = q[st] - qr[k];
                    ++j;
                }
                plm_inc64<2 * N>(lo, hi, t);
#pragma unroll
                for (int k = 0, j = 0; k < NV; ++k) {
                    if (MHD && k == BCC) continue;
                    ql[k] += t[j];
                    qr[k] -= t[N + j];
                    ++j;
                }
            }
            if constexpr (MHD) {
                const int p[3] = {gx, gy, 0};
                const FT bn = xf ? (FT)load_bf(m, b, step, 0, p) : (FT)load_bf(m, b, step, 1, p);
                ql[BCC] = bn;
                qr[BCC] = bn;
                if constexpr (std::is_same_v<FT, float>) hlld_fast(flx, ql, qr, (FT)m.gamma);
                else hlld64(flx, ql, qr, Gam64{m.gamma, m.cv, m.ge});
            } else {
                if constexpr (std::is_same_v<FT, float>) hllc_fast(flx, ql, qr, (FT)m.gamma);
                else hllc64(flx, ql, qr, Gam64{m.gamma, m.cv, m.ge});
            }
            sF[RHO][tid] = flx[RHO];
            sF[ENE][tid] = flx[ENE];
            sF[MOM][tid] = xf ? flx[MOM] : flx[MOM + 2];
            sF[MOM + 1][tid] = xf ? flx[MOM + 1] : flx[MOM];
            sF[MOM + 2][tid] = xf ? flx[MOM + 2] : flx[MOM + 1];
            if constexpr (MHD) {
                // x faces: E_y, E_z; y faces: E_x, E_z
                sE[0][tid] = xf ? flx[BCC + 2] : -flx[BCC + 1];
                sE[1][tid] = xf ? -flx[BCC + 1] : flx[BCC + 2];
            }
        }
    }
    __syncthreads();

    // ---------------------------------------------- edge EMFs
    const int px = tid % (TX + 1), py = tid / (TX + 1);
    const int gx = x0 + px, gy = y0 + py;
    // points of the tile: its cells, and the block's high faces next to them
    const bool point = tid < NP && gx <= n0 && gy <= n1;
    if constexpr (MHD) {
        if (point) {
            auto ec = [&](int x, int y, int c) -> FT {
                const int cc = col(x, y);
                const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
                return sW[BCC + c1][cc] * sW[MOM + c2][cc] - sW[BCC + c2][cc] * sW[MOM + c1][cc];
            };
            // an edge next to a thin axis takes the surviving sweep's face
            // value (integrator.h:221-300)
            FT e[3] = {0, 0, 0};
            if constexpr (two) {
                if (gx < n0) e[0] = sE[0][fyi(px, py)];
                if (gy < n1) e[1] = sE[0][fxi(px, py)];
                e[2] = corner_emf<FT>(ec(px, py, 2), ec(px - 1, py, 2), ec(px - 1, py - 1, 2), ec(px, py - 1, 2),
                                      sE[1][fxi(px, py - 1)], sE[1][fxi(px, py)], sF[RHO][fyi(px, py)],
                                      sF[RHO][fyi(px - 1, py)], sE[1][fyi(px - 1, py)], sE[1][fyi(px, py)],
                                      sF[RHO][fxi(px, py)], sF[RHO][fxi(px, py - 1)]);
            } else {
                e[1] = sE[0][fxi(px, 0)];
                e[2] = sE[1][fxi(px, 0)];
            }
            if (g.phy) {
                // boundary-plane EMF of a high out / fre side (as in k_emf)
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    const int i = a == 0 ? gx : gy;
                    if (i != m.n[a] || m.n[a] < 2 || !((g.phy >> (2 * a + 1)) & 1)) continue;
                    const int k = m.bnd[2 * a + 1];
                    if (k != 1 && k != 2) continue;
                    const int cc = col(px - (a == 0), py - (a == 1));
                    const FT irho = (FT)1 / pmax(sW[RHO][cc], (FT)1e-30);
                    FT v_c[3], b_c[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        v_c[q] = sW[MOM + q][cc] * irho;
                        b_c[q] = sW[BCC + q][cc];
                    }
                    const int a1 = a + 1, a2 = a == 0 ? 2 : 0;
                    e[a1] = v_c[a] * b_c[a2] - v_c[a2] * b_c[a];
                    e[a2] = v_c[a1] * b_c[a] - v_c[a] * b_c[a1];
                }
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) sEd[q][edi(px, py)] = e[q];
        }
        __syncthreads();
    }

    // ---------------------------------------------- update
    if (point && px < TX && py < TY && gx < n0 && gy < n1) {
        const size_t c = cidx(m.n, gx, gy, 0);
        const double *Us = m.U + ((size_t)b * 2 + step) * 5 * nc + c;
        double *Ut = m.U + ((size_t)b * 2 + (1 - step)) * 5 * nc + c;
        double uu[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) uu[v] = Us[(size_t)v * nc];
        if constexpr (C2P) {
            uu[RHO] = sU[0][py * TX + px];
            uu[ENE] = sU[1][py * TX + px];
        }
        if (step != 0) {
#pragma unroll
            for (int v = 0; v < 5; ++v) uu[v] = (uu[v] + Ut[(size_t)v * nc]) * 0.5f;
        }
        const double dt_dv = dt / g.vol;
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            if (a == 1 && !two) continue;
            const int i0 = a == 0 ? fxi(px, py) : fyi(px, py);
            const int i1 = a == 0 ? fxi(px + 1, py) : fyi(px, py + 1);
            const FT fa = (FT)(g.sfc[a] * dt_dv);
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                double res(0);
                if (fa > 0) res += (double)(fa * sF[v][i0]);
                if (fa > 0) res -= (double)(fa * sF[v][i1]);
                uu[v] += res;
            }
        }
#pragma unroll
        for (int v = 0; v < 5; ++v) Ut[(size_t)v * nc] = uu[v];
    }
    if constexpr (MHD) {
        if (point) {
            // a point past the tile is this tile's only at the block's end
            const bool mx = px < TX || gx == n0, my = py < TY || gy == n1;
            const size_t f = fidx(m.n, gx, gy, 0);
            const double *Bs = m.BF + ((size_t)b * 2 + step) * 3 * m.nface + f;
            double *Bt = m.BF + ((size_t)b * 2 + (1 - step)) * 3 * m.nface + f;
            auto put = [&](int a, double db, double sfc) {
                db *= (sfc > 0 ? (double)(-dt / sfc) : (double)(0));
                const double bs = Bs[(size_t)a * m.nface];
                Bt[(size_t)a * m.nface] = db + (step == 0 ? bs : (bs + Bt[(size_t)a * m.nface]) / 2);
            };
            const int e = edi(px, py), ex = edi(px + 1, py), ey = edi(px, py + 1);
            const double dx = g.dx[0], dy = g.dx[1], dz = g.dx[2];
            // mhd/integrator/integrator.h:385-462; an edge pair spanning a thin
            // axis vanishes (:419-447)
            if (mx && py < TY && gy < n1) {
                double db = 0.0;
                if (two) {
                    db -= (double)sEd[2][e] * dz;
                    db += (double)sEd[2][ey] * dz;
                }
                put(0, db, g.sfc[0]);
            }
            if (my && px < TX && gx < n0) {
                double db = (double)sEd[2][e] * dz;
                db -= (double)sEd[2][ex] * dz;
                put(1, db, two ? g.sfc[1] : dz * dx);
            }
            if (px < TX && py < TY && gx < n0 && gy < n1) {
                double db = two ? (double)sEd[0][e] * dx : 0.0;
                db -= (double)sEd[1][e] * dy;
                db += (double)sEd[1][ex] * dy;
                if (two) db -= (double)sEd[0][ey] * dx;
                put(2, db, dx * dy);
            }
        }
    }
}

}  // namespace kr
