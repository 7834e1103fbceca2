// kr_march.h -- fused MHD stage kernel: the z march, LDS ring, edge EMFs,
// update and constrained transport of k_sweep (kr_fused.h), with the Riemann
// solves of a plane spread evenly over the waves, for blocks of any size from
// one tile up.  It runs the FP64 form, and the mixed form (FP32 fluxes, FP64
// state) on blocks that k_sweep_mx's tiles do not divide.
//
// The FP64 solves bound the kernel: a second workgroup on a compute unit
// gains nothing (time follows the workgroups per compute unit), so what
// counts is the wave that solves most.  Giving z pencils, x faces and y faces
// waves of their own leaves a 16x8 tile with 9 waves of solves on 4 waves:
// three on one SIMD, two on the others.  Here a plane's solves are one list,
//   [z faces of the owned columns][z faces of the columns around][x][y],
// walked in rounds of the workgroup through one call of the solver: 508 items
// of a 16x8 tile are two rounds of 256 threads, 972 of 32x8 two of 512.  The
// owned columns' z pencils keep their state in registers (they are the first
// round's first waves); the columns around, which only feed the EMFs, keep
// their left state in LDS.  The per-face arithmetic and its order are those
// of the staged kernels (kr_exact64.h in FP64), so the results equal theirs,
// and in FP64 the oracle's, bit for bit.
//
// Where the tile does not divide the block, its last tile along an axis is
// moved back into the block and shares columns with the one before: both
// compute them, the one before stores them.  The shared columns and the
// staged kernels' five launches cost about the same where the tiles fill the
// GPU (300,000 cells in 20x12x25 blocks, mixed: 254 against 256 us a cycle),
// so the tuner times both there; on fewer cells the march wins (12,000 cells:
// 95 against 117 us), as on blocks a little larger than its tiles (24^3 in
// 96^3, FP64: 739 against 903 us).
#pragma once

#include "kr_exact64.h"
#include "kr_fused.h"

namespace kr {

template <int TX, int TY>
struct Tile64 {
    using S = TileShape<TX, TY>;
    static constexpr int NZ = TX * TY;                        // owned columns
    static constexpr int NRING = 2 * (TX + TY);               // columns around, without corners
    static constexpr int NITEM = NZ + NRING + S::NFX + S::NFY;
    // faces of the tile itself (no transverse ghost lines)
    static constexpr int NIX = (TX + 1) * TY, NIY = TX * (TY + 1), NI = NIX + NIY;
    __device__ static int ix(int x, int y) { return y * (TX + 1) + x; }
    __device__ static int iy(int x, int y) { return NIX + y * TX + x; }
};

// Workgroups along an axis of n cells.
__host__ __device__ inline int march_tiles(int n, int t) { return (n + t - 1) / t; }

// PROD = 1 (refined meshes, blocks that touch another level): the kernel only
// produces the fluxes (F) and edge EMFs (EE) of the block, as k_sweep's
// producer form does.  PHY: meshes with physical sides.
template <class FT, int TX, int TY, int NT, int PROD = 0, bool PHY = false>
__global__ void __launch_bounds__(NT) k_march(MeshView<FT> m, int step) {
    constexpr bool F32 = std::is_same_v<FT, float>;
    using S = TileShape<TX, TY>;
    using T = Tile64<TX, TY>;
    constexpr int NROUND = (T::NITEM + NT - 1) / NT;
    static_assert(T::NZ <= NT && T::NZ % 64 == 0, "owned columns: whole waves of the first round");
    static_assert(TX * TY + TX + TY <= NT, "one owned cell / edge face per thread");
    unsigned tile, row;
    xcd_tile(tile, row);
    const int b = m.blist ? m.blist[row] : (int)row;
    if (m.ts[m.geo[b].grp].skip) return;
    const int tid = threadIdx.x;
    const int ntx = march_tiles(m.n[0], TX);
    const int xs = (tile % ntx) * TX, ys = (tile / ntx) * TY;
    // first column and row of the tile, and of its own cells in it
    const int x0 = xs + TX > m.n[0] ? m.n[0] - TX : xs, y0 = ys + TY > m.n[1] ? m.n[1] - TY : ys;
    const int ox = xs - x0, oy = ys - y0;
    const int nz = m.n[2];
    int z0, z1;
    z_range(nz, z0, z1);
    const bool xlast = x0 + TX == m.n[0], ylast = y0 + TY == m.n[1];
    const BlockGeo &g = m.geo[b];
    const double dt = m.ts[g.grp].dt_use * (step == 0 ? 1.0 : 0.5);
    const size_t nc = m.ncell;
    const Gam64 gam{m.gamma, m.cv, m.ge};

    constexpr int DPC = (int)sizeof(FT) / 4;                       // dwords per column
    constexpr int NDW = S::NCOL * DPC;                             // dwords per row
    constexpr int NCHUNK = (NDW + 63) / 64;                        // chunks per row
    __shared__ FT sW[3][8][S::NCOL];
    __shared__ FT sFr[2][S::NF];        // in-plane faces of two planes: mass flux ...
    __shared__ FT sFt[2][T::NI];        // ... and E_y of x faces, E_x of y faces
    __shared__ FT sFez[S::NF];          // E_z of the current plane's faces
    __shared__ FT sFh[4][T::NI];        // their energy and momentum fluxes
    __shared__ FT sFz[3][S::NZG];       // rho, E_x, E_y of the current z face
    __shared__ FT sEz[2][S::NEZ];
    __shared__ FT sEx[2][S::NEX];
    __shared__ FT sEy[2][S::NEY];
    __shared__ FT sQ[7][T::NRING];      // left states of the columns around
    __shared__ int sNbr[27];
    __shared__ double sGeo[9];          // -dt / sfc_a, sfc_a dt / vol, dx_a
    if (tid < 27) sNbr[tid] = g.wnbr[tid];
    if (tid < 3) {
        const double sfc = g.sfc[tid];
        sGeo[tid] = sfc > 0 ? (double)(-dt / sfc) : (double)(0);
        sGeo[3 + tid] = sfc * (dt / g.vol);
        sGeo[6 + tid] = g.dx[tid];
    }
    __syncthreads();

    // primitive source of halo column (cx, cy) at plane z
    auto wsrc = [&](int cx, int cy, int z) -> const FT * {
        int p[3] = {x0 + cx, y0 + cy, z};
        int d[3];
        bool out = false;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            d[a] = p[a] < 0 ? -1 : (p[a] >= m.n[a] ? 1 : 0);
            out |= d[a] != 0;
        }
        int blk = b;
        if (out) {
            blk = sNbr[((d[2] + 1) * 3 + (d[1] + 1)) * 3 + (d[0] + 1)];
#pragma unroll
            for (int a = 0; a < 3; ++a) p[a] -= d[a] * m.n[a];
        }
        return m.W + (size_t)blk * 8 * nc + cidx(m.n, p[0], p[1], p[2]);
    };
    // normal face field of face (fx, fy, fz), component c (see k_sweep's bfn:
    // the same rules at physical sides and next to another level)
    auto bfn = [&](int c, int fx, int fy, int fz, int slot) -> FT {
        int p[3] = {x0 + fx, y0 + fy, fz};
        int d[3] = {0, 0, 0};
        bool out = false;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (a == c) continue;
            d[a] = p[a] < 0 ? -1 : (p[a] >= m.n[a] ? 1 : 0);
            out |= d[a] != 0;
        }
        int blk = b;
        if (PHY && out && g.phy) {
            int a = 0;
#pragma unroll
            for (int x = 0; x < 3; ++x)
                if (d[x]) a = x;
            int da = 0;
#pragma unroll
            for (int x = 0; x < 3; ++x)
                if (x == a) da = d[x];
            if ((g.phy >> (2 * a + (da > 0))) & 1) {
                const int side = da > 0;
                const int kind = m.bnd[2 * a + side];
                if (kind == 4) return (FT)(c == 0 ? m.fix_b[0] : (c == 1 ? m.fix_b[1] : m.fix_b[2]));
                double sgn = 1;
                const bool top = (g.phy >> (2 * c + 1)) & 1;
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    if (x == a) {
                        if (kind == 3) {
                            p[x] = side ? m.n[x] - 2 : 1;
                            sgn = -1;
                        } else {
                            p[x] = side ? m.n[x] - 1 : 0;
                        }
                    }
                    if (x == c && top && p[x] >= m.n[x]) p[x] = m.n[x] - 1;
                }
                return (FT)(sgn * m.BF[(((size_t)b * 2 + step) * 3 + c) * m.nface +
                                       fidx(m.n, p[0], p[1], p[2])]);
            }
        }
        if constexpr (PROD) {
            if (out && g.xface) {
                int bit = 0;
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    if (d[a]) bit = 1 << (2 * a + (d[a] > 0));
                if (g.xface & bit) return sW[slot][BCC + c][S::col(fx, fy)];
            }
        }
        if (out) {
            blk = sNbr[((d[2] + 1) * 3 + (d[1] + 1)) * 3 + (d[0] + 1)];
#pragma unroll
            for (int a = 0; a < 3; ++a) p[a] -= d[a] * m.n[a];
        }
        return (FT)m.BF[(((size_t)blk * 2 + step) * 3 + c) * m.nface + fidx(m.n, p[0], p[1], p[2])];
    };
    // asynchronous load of plane z of W into ring slot `slot`
    auto issue_w = [&](int z, int slot) {
        const int wave = tid >> 6, lane = tid & 63;
        for (int k = wave; k < NCHUNK; k += NT / 64) {
            const int d = k * 64 + lane;
            if (d >= NDW) continue;                 // past the row: no load, no write
            const int col = d / DPC;
            const int half = d - col * DPC;
            const FT *src = wsrc(col % S::HX - 2, col / S::HX - 2, z);
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                const char *gp = (const char *)(src + (size_t)v * nc) + 4 * half;
                __builtin_amdgcn_global_load_lds(gp, &sW[slot][v][0] + k * (64 / DPC), 4, 0, 0);
            }
        }
    };

    // owned column of the first NZ threads
    const int cx_ = tid < T::NZ ? tid % TX : 0, cy_ = tid < T::NZ ? tid / TX : 0;
    const bool zint = tid < T::NZ && cx_ >= ox && cy_ >= oy;
    FT qL[7];                 // left state of the next z face, z frame
    FT fzp[5];                // hydro z flux of the previous face
    double part[5];           // x + y partial update of the previous plane
#pragma unroll
    for (int v = 0; v < 7; ++v) qL[v] = 0;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        fzp[v] = 0;
        part[v] = 0;
    }
    // high sides of the block: threads TX*TY .. +TY-1 own the x faces at
    // x = TX, the next TX threads the y faces at y = TY
    const int et = tid - TX * TY;
    const bool xedge = xlast && et >= oy && et < TY;
    const bool yedge = ylast && et >= TY + ox && et < TY + TX;

    issue_w(z0 - 2, ring3(z0 - 2));
    for (int L = z0 - 2; L <= z1 + 1; ++L) {
        // ------------------------------------------------ 1. plane L arrives
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        const int P = L - 2;          // plane finished in this iteration

        // ------------------------------------------------ 2. fluxes
        if (L >= z0) {
            const int p = L - 1;                 // plane of the in-plane faces / z face index
            const int s0 = ring3(p), sm = ring3(p - 1), sp = ring3(p + 1);
            const int fe = ring2(p);
            const bool ghost_plane = p < 0 || p >= nz;
#pragma unroll 1
            for (int r = 0; r < NROUND; ++r) {
                const int it = r * NT + tid;
                if (it >= T::NITEM) break;
                // the item's axis a and face (fx, fy), z faces at index p
                int a, fx, fy, ri = 0;
                if (it < T::NZ) {
                    a = 2;
                    fx = it % TX;
                    fy = it / TX;
                } else if (it < T::NZ + T::NRING) {
                    a = 2;
                    ri = it - T::NZ;
                    if (ri < 2 * TX) {
                        fx = ri % TX;
                        fy = ri < TX ? -1 : TY;
                    } else {
                        fx = ri < 2 * TX + TY ? -1 : TX;
                        fy = (ri - 2 * TX) % TY;
                    }
                } else if (it < T::NZ + T::NRING + S::NFX) {
                    const int k = it - T::NZ - T::NRING;
                    a = 0;
                    fx = k % (TX + 1);
                    fy = k / (TX + 1) - 1;
                } else {
                    const int k = it - T::NZ - T::NRING - S::NFX;
                    a = 1;
                    fx = k % (TX + 2) - 1;
                    fy = k / (TX + 2);
                }
                // face of the tile itself, not of a transverse ghost line
                const bool inner = a == 0 ? (fy >= 0 && fy < TY) : (fx >= 0 && fx < TX);
                if (a < 2 && ghost_plane && !inner) continue;
                const FT bn = a == 0 ? bfn(0, fx, fy, p, s0)
                                     : (a == 1 ? bfn(1, fx, fy, p, s0) : (p >= z0 ? bfn(2, fx, fy, p, s0) : 0));
                FT wl[8], wr[8], flx[8];
                if (it < T::NZ) {
                    // an owned column's z pencil (whole waves)
                    const FT *q = &sW[0][0][S::col(fx, fy)];
                    constexpr int PL = 8 * S::NCOL;
                    constexpr int slot[7] = {RHO, ENE, MOM, MOM + 1, MOM + 2, BCC + 1, BCC + 2};
                    constexpr int vz[7] = {RHO, ENE, MOM + 2, MOM, MOM + 1, BCC, BCC + 1};
                    FT c[7], lo[7], hi[7], t[7];
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        const int v = vz[j] * S::NCOL;
                        c[j] = q[s0 * PL + v];
                        lo[j] = c[j] - q[sm * PL + v];
                        hi[j] = q[sp * PL + v] - c[j];
                    }
                    if constexpr (F32) {
#pragma unroll
                        for (int j = 0; j < 7; ++j) {
                            const int v = vz[j] * S::NCOL;
                            t[j] = plm_inc_fast(q[sm * PL + v], c[j], q[sp * PL + v]);
                        }
                    } else {
                        plm_inc64<7>(lo, hi, t);
                    }
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        wl[slot[j]] = qL[j];
                        wr[slot[j]] = c[j] - t[j];
                        qL[j] = c[j] + t[j];
                    }
                } else {
                    // right cell of the face and its neighbours along the axis; a z
                    // face's left state is what the plane before left in sQ
                    const FT *q0p = &sW[s0][0][S::col(fx, fy)];
                    const int om = a == 0 ? -1 : (a == 1 ? -S::HX : (sm - s0) * 8 * S::NCOL);
                    const int op = a == 0 ? 1 : (a == 1 ? S::HX : (sp - s0) * 8 * S::NCOL);
                    const int om2 = a == 2 ? om : 2 * om;
                    // rotated frame: slot k holds mesh variable perm(k); the
                    // normal field (slot BCC) comes from the face
                    const int r0 = a * S::NCOL, r1 = (a == 2 ? 0 : a + 1) * S::NCOL,
                              r2 = (a == 0 ? 2 : a - 1) * S::NCOL;
                    constexpr int slot[7] = {RHO, ENE, MOM, MOM + 1, MOM + 2, BCC + 1, BCC + 2};
                    const int off[7] = {RHO * S::NCOL, ENE * S::NCOL, MOM * S::NCOL + r0, MOM * S::NCOL + r1,
                                        MOM * S::NCOL + r2, BCC * S::NCOL + r1, BCC * S::NCOL + r2};
                    FT c[7], ql[7], lo[14], hi[14], t[14];
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        const FT *q = q0p + off[j];
                        c[j] = q[0];
                        ql[j] = q[om];
                        if constexpr (F32) {
                            t[j] = plm_inc_fast(ql[j], c[j], q[op]);
                            t[7 + j] = plm_inc_fast(q[om2], ql[j], c[j]);
                        } else {
                            lo[j] = c[j] - ql[j];
                            hi[j] = q[op] - c[j];
                            lo[7 + j] = ql[j] - q[om2];
                            hi[7 + j] = lo[j];
                        }
                    }
                    if constexpr (!F32) plm_inc64<14>(lo, hi, t);
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        const FT wq = sQ[j][ri];
                        wr[slot[j]] = c[j] - t[j];
                        wl[slot[j]] = a == 2 ? wq : ql[j] + t[7 + j];
                        if (a == 2) sQ[j][ri] = c[j] + t[j];
                    }
                }
                if (a == 2 && p < z0) continue;      // a range's lead-in cell
                wl[BCC] = bn;
                wr[BCC] = bn;
                if constexpr (F32) hlld_fast(flx, wl, wr, (FT)m.gamma);
                else hlld64(flx, wl, wr, gam);
                if (a == 2) {
                    // rotated frame (z, x, y): E_x = flx[B_y], E_y = -flx[B_x]
                    const int gz = S::zg(fx, fy);
                    sFz[0][gz] = flx[RHO];
                    sFz[1][gz] = flx[BCC + 2];
                    sFz[2][gz] = -flx[BCC + 1];
                    const FT f[5] = {flx[RHO], flx[ENE], flx[MOM + 1], flx[MOM + 2], flx[MOM]};
                    if (it < T::NZ) {
                        if constexpr (PROD) {
                            if (p < z1 || z1 == nz) {
                                const int q3[3] = {x0 + fx, y0 + fy, p};
                                FT *F = m.F[2] + (size_t)b * 8 * m.nfa[2] + xidx(m.n, 2, q3);
#pragma unroll
                                for (int v = 0; v < 5; ++v) F[(size_t)v * m.nfa[2]] = f[v];
                            }
                        } else {
                            // z part of the cell finished now (plane P)
                            if (P >= z0 && zint) {
                                const FT fa = (FT)sGeo[3 + 2];
                                double *Ut = m.U + ((size_t)b * 2 + (1 - step)) * 5 * nc +
                                             cidx(m.n, x0 + fx, y0 + fy, P);
#pragma unroll
                                for (int v = 0; v < 5; ++v) {
                                    double res(0);
                                    if (fa > 0) res += (double)(fa * fzp[v]);
                                    if (fa > 0) res -= (double)(fa * f[v]);
                                    Ut[(size_t)v * nc] = part[v] + res;
                                }
                            }
#pragma unroll
                            for (int v = 0; v < 5; ++v) fzp[v] = f[v];
                        }
                    }
                } else {
                    const bool xf = a == 0;
                    const int e = xf ? S::fxi(fx, fy) : S::fyi(fx, fy);
                    // x faces: E_y, E_z; y faces: E_x, E_z
                    const FT et1 = xf ? flx[BCC + 2] : -flx[BCC + 1];
                    sFr[fe][e] = flx[RHO];
                    sFez[e] = xf ? -flx[BCC + 1] : flx[BCC + 2];
                    if (inner) {
                        const int i = xf ? T::ix(fx, fy) : T::iy(fx, fy);
                        const FT mx = xf ? flx[MOM] : flx[MOM + 2], my = xf ? flx[MOM + 1] : flx[MOM],
                                 mz = xf ? flx[MOM + 2] : flx[MOM + 1];
                        sFt[fe][i] = et1;
                        if constexpr (PROD) {
                            if (p >= z0 && p < z1) {
                                const int q3[3] = {x0 + fx, y0 + fy, p};
                                const size_t nf = xf ? m.nfa[0] : m.nfa[1];
                                FT *F = (xf ? m.F[0] : m.F[1]) + (size_t)b * 8 * nf +
                                        (xf ? xidx(m.n, 0, q3) : xidx(m.n, 1, q3));
                                F[(size_t)RHO * nf] = flx[RHO];
                                F[(size_t)ENE * nf] = flx[ENE];
                                F[(size_t)MOM * nf] = mx;
                                F[(size_t)(MOM + 1) * nf] = my;
                                F[(size_t)(MOM + 2) * nf] = mz;
                            }
                        } else {
                            sFh[0][i] = flx[ENE];
                            sFh[1][i] = mx;
                            sFh[2][i] = my;
                            sFh[3][i] = mz;
                        }
                    }
                }
            }
        }
        __syncthreads();

        // ------------------------------------------------ 3. EMFs
        if (L >= z0 + 1) {
            const int p = L - 1;
            const bool own_p = p < z1 || z1 == nz;
            const int s0 = ring3(p), sm = ring3(p - 1);
            const int fe = ring2(p), fm = ring2(p - 1);
            auto ec = [&](int s, int x, int y, int c) -> FT {
                const int cc = S::col(x, y);
                const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
                const FT b1 = sW[s][BCC + c1][cc], v2 = sW[s][MOM + c2][cc];
                const FT b2 = sW[s][BCC + c2][cc], v1 = sW[s][MOM + c1][cc];
                return b1 * v2 - b2 * v1;
            };
            // boundary-plane EMF of a high out / fre side (as in k_sweep)
            auto bplane = [&](int c, int x, int y, FT e) -> FT {
                const int gi[3] = {x0 + x, y0 + y, p};
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    if (a == c || gi[a] != m.n[a] || m.n[a] < 2 || !((g.phy >> (2 * a + 1)) & 1)) continue;
                    const int k = m.bnd[2 * a + 1];
                    if (k != 1 && k != 2) continue;
                    const int cc = S::col(x - (a == 0), y - (a == 1));
                    const int sl = a == 2 ? sm : s0;
                    FT w[8];
#pragma unroll
                    for (int v = 0; v < 8; ++v) w[v] = sW[sl][v][cc];
                    const FT irho = (FT)1 / pmax(w[RHO], (FT)1e-30);
                    FT v_c[3], b_c[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        v_c[q] = w[MOM + q] * irho;
                        b_c[q] = w[BCC + q];
                    }
                    const int a1 = mod3(a + 1), a2 = mod3(a + 2);
                    if (c == a1) e = v_c[a] * b_c[a2] - v_c[a2] * b_c[a];
                    else e = v_c[a1] * b_c[a] - v_c[a] * b_c[a1];
                }
                return e;
            };
            for (int it = tid; it < S::NEZ + S::NEX + S::NEY; it += NT) {
                if (it < S::NEZ) {
                    if (p >= z1) continue;
                    const int x = it % (TX + 1), y = it / (TX + 1);
                    // ee_z on plane p: a1 = x, a2 = y
                    FT e = corner_emf<FT>(
                        ec(s0, x, y, 2), ec(s0, x - 1, y, 2), ec(s0, x - 1, y - 1, 2), ec(s0, x, y - 1, 2),
                        sFez[S::fxi(x, y - 1)], sFez[S::fxi(x, y)], sFr[fe][S::fyi(x, y)],
                        sFr[fe][S::fyi(x - 1, y)], sFez[S::fyi(x - 1, y)], sFez[S::fyi(x, y)],
                        sFr[fe][S::fxi(x, y)], sFr[fe][S::fxi(x, y - 1)]);
                    if (PHY && g.phy) e = bplane(2, x, y, e);
                    sEz[fe][S::ezi(x, y)] = e;
                    if constexpr (PROD)
                        m.EE[((size_t)b * 3 + 2) * m.nface + fidx(m.n, x0 + x, y0 + y, p)] = e;
                } else if (it < S::NEZ + S::NEX) {
                    const int k = it - S::NEZ;
                    const int x = k % TX, y = k / TX;
                    // ee_x on z face p: a1 = y, a2 = z
                    FT e = corner_emf<FT>(
                        ec(s0, x, y, 0), ec(s0, x, y - 1, 0), ec(sm, x, y - 1, 0), ec(sm, x, y, 0),
                        sFt[fm][T::iy(x, y)], sFt[fe][T::iy(x, y)], sFz[0][S::zg(x, y)],
                        sFz[0][S::zg(x, y - 1)], sFz[1][S::zg(x, y - 1)], sFz[1][S::zg(x, y)],
                        sFr[fe][S::fyi(x, y)], sFr[fm][S::fyi(x, y)]);
                    if (PHY && g.phy) e = bplane(0, x, y, e);
                    sEx[fe][S::exi(x, y)] = e;
                    if (PROD && own_p)
                        m.EE[((size_t)b * 3 + 0) * m.nface + fidx(m.n, x0 + x, y0 + y, p)] = e;
                } else {
                    const int k = it - S::NEZ - S::NEX;
                    const int x = k % (TX + 1), y = k / (TX + 1);
                    // ee_y on z face p: a1 = z, a2 = x
                    FT e = corner_emf<FT>(
                        ec(s0, x, y, 1), ec(sm, x, y, 1), ec(sm, x - 1, y, 1), ec(s0, x - 1, y, 1),
                        sFz[2][S::zg(x - 1, y)], sFz[2][S::zg(x, y)], sFr[fe][S::fxi(x, y)],
                        sFr[fm][S::fxi(x, y)], sFt[fm][T::ix(x, y)], sFt[fe][T::ix(x, y)],
                        sFz[0][S::zg(x, y)], sFz[0][S::zg(x - 1, y)]);
                    if (PHY && g.phy) e = bplane(1, x, y, e);
                    sEy[fe][S::eyi(x, y)] = e;
                    if (PROD && own_p)
                        m.EE[((size_t)b * 3 + 1) * m.nface + fidx(m.n, x0 + x, y0 + y, p)] = e;
                }
            }
        }
        __syncthreads();

        // plane L+1 into the slot of plane L-2, which phases 2 and 3 of this
        // iteration were the last to read; it lands while the update runs
        if (L + 1 <= z1 + 1) issue_w(L + 1, ring3(L + 1));

        // ------------------------------------------------ 4. update
        if (!PROD && L >= z0 + 1) {
            const int q = L - 1;                     // z face updated now
            const int fq = ring2(q), fpp = ring2(P);
            // a face's two slots are read first, with the conserved state, and
            // written last, so that the loads are in flight together
            struct FaceUpd {
                double *bt;
                double s, t;
            };
            auto face_load = [&](int c, int fx, int fy, int fz) {
                const size_t f = fidx(m.n, x0 + fx, y0 + fy, fz);
                FaceUpd u;
                u.bt = m.BF + (((size_t)b * 2 + (1 - step)) * 3 + c) * m.nface + f;
                u.s = m.BF[(((size_t)b * 2 + step) * 3 + c) * m.nface + f];
                u.t = step == 0 ? 0.0 : *u.bt;
                return u;
            };
            auto face_store = [&](const FaceUpd &u, double db) {
                *u.bt = db + (step == 0 ? u.s : (u.s + u.t) / 2);
            };
            // CT circulation of one face (mhd/integrator/integrator.h:429-457)
            auto ct = [&](double e1, double d1, double e2, double d2, double e3, double e4, int a) {
                double db = e1 * d1;
                db -= e2 * d2;
                db += e3 * d2;
                db -= e4 * d1;
                db *= sGeo[a];
                return db;
            };
            const double dx = sGeo[6], dy = sGeo[7], dz = sGeo[8];
            if (zint) {
                const int x = cx_, y = cy_;
                const FaceUpd uz = face_load(2, x, y, q);
                const FaceUpd ux = face_load(0, x, y, P < z0 ? z0 : P);
                const FaceUpd uy = face_load(1, x, y, P < z0 ? z0 : P);
                // x + y partial of plane q (cells), finished next iteration
                if (q < z1) {
                    const size_t c = cidx(m.n, x0 + x, y0 + y, q);
                    const double *Us = m.U + ((size_t)b * 2 + step) * 5 * nc + c;
                    const double *Ut = m.U + ((size_t)b * 2 + (1 - step)) * 5 * nc + c;
                    double uu[5];
                    if (step == 0) {
#pragma unroll
                        for (int v = 0; v < 5; ++v) uu[v] = Us[(size_t)v * nc];
                    } else {
#pragma unroll
                        for (int v = 0; v < 5; ++v) uu[v] = (Us[(size_t)v * nc] + Ut[(size_t)v * nc]) * 0.5f;
                    }
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        const int e0 = a == 0 ? S::fxi(x, y) : S::fyi(x, y);
                        const int e1 = a == 0 ? S::fxi(x + 1, y) : S::fyi(x, y + 1);
                        const int i0 = a == 0 ? T::ix(x, y) : T::iy(x, y);
                        const int i1 = a == 0 ? T::ix(x + 1, y) : T::iy(x, y + 1);
                        const FT fa = (FT)sGeo[3 + a];
#pragma unroll
                        for (int v = 0; v < 5; ++v) {
                            double res(0);
                            const FT f0 = v == 0 ? sFr[fq][e0] : sFh[v - 1][i0];
                            const FT f1 = v == 0 ? sFr[fq][e1] : sFh[v - 1][i1];
                            if (fa > 0) res += (double)(fa * f0);
                            if (fa > 0) res -= (double)(fa * f1);
                            uu[v] += res;
                        }
                    }
#pragma unroll
                    for (int v = 0; v < 5; ++v) part[v] = uu[v];
                }
                // z face q: the range's own faces, and the block's top face in
                // the last range
                if (q < z1 || z1 == nz)
                    face_store(uz, ct(sEx[fq][S::exi(x, y)], dx, sEy[fq][S::eyi(x, y)], dy,
                                      sEy[fq][S::eyi(x + 1, y)], sEx[fq][S::exi(x, y + 1)], 2));
                if (P >= z0) {
                    face_store(ux, ct(sEy[fpp][S::eyi(x, y)], dy, sEz[fpp][S::ezi(x, y)], dz,
                                      sEz[fpp][S::ezi(x, y + 1)], sEy[fq][S::eyi(x, y)], 0));
                    face_store(uy, ct(sEz[fpp][S::ezi(x, y)], dz, sEx[fpp][S::exi(x, y)], dx,
                                      sEx[fq][S::exi(x, y)], sEz[fpp][S::ezi(x + 1, y)], 1));
                }
            }
            if (P >= z0 && xedge) {
                const int x = TX, y = et;
                const FaceUpd ux = face_load(0, x, y, P);
                face_store(ux, ct(sEy[fpp][S::eyi(x, y)], dy, sEz[fpp][S::ezi(x, y)], dz,
                                  sEz[fpp][S::ezi(x, y + 1)], sEy[fq][S::eyi(x, y)], 0));
            }
            if (P >= z0 && yedge) {
                const int x = et - TY, y = TY;
                const FaceUpd uy = face_load(1, x, y, P);
                face_store(uy, ct(sEz[fpp][S::ezi(x, y)], dz, sEx[fpp][S::exi(x, y)], dx,
                                  sEx[fq][S::exi(x, y)], sEz[fpp][S::ezi(x + 1, y)], 1));
            }
        }
    }
}

}  // namespace kr
