// kr_pack.h -- a block's state between the pools (SoA, one plane per
// variable) and the reference's host layout (AoS, ghosted faces), and the
// time states, through page-locked host memory that the kernels address
// directly.
//
// Repacking on the host took most of a transfer: two copies by the runtime,
// two vectors and three strided loops over each block (128 MHD blocks of 8^3:
// 35 us a block).  Here one thread moves one double of the host arrays, with
// consecutive threads on consecutive doubles, so the bus sees full lines;
// what is left on the host is one contiguous copy per array.  (Small hydro
// blocks, one range and no faces, are transposed on the host: kr_api.hip.)
#pragma once

#include "kr_staged.h"

namespace kr {

// Host arrays of a block: u (ncell * nvar), then for MHD the face array with
// two ghost layers a side, N[a] = n[a] + (n[a] > 1) + 4.  Of that one the
// doubles from the block's first face to its last are moved, bf0 .. bf0 + nbf:
// the ghost layers before and behind are not read, and zeros on the way back
// (four fifths of a 2-D block's array, 24 of 25 rows of a 1-D block's).
struct HostShape {
    int n[3], N[3], nvar;
    size_t nu, bf0, nbf;     // doubles of u, first and number of those of bf
};

// Doubles [i0, i0 + count) of what is moved of a block's host arrays (u, then
// bf) into out, from slot 0: u's cell-centred B is the face average, ghost
// faces are 0.
__global__ void __launch_bounds__(kThreads) k_pack(HostShape h, const double *U, const double *BF,
                                                   size_t ncell, size_t nface, size_t i0, size_t count,
                                                   double *out) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const size_t i = i0 + t;
    const int nx = h.n[0] + 1, nxy = nx * (h.n[1] + 1);
    double v = 0;
    if (i < h.nu) {
        const unsigned c = (unsigned)(i / h.nvar);
        const int k = (int)(i - (size_t)c * h.nvar);
        if (k < 5) {
            v = U[(size_t)k * ncell + c];
        } else {
            const unsigned x = c % h.n[0], r = c / h.n[0];
            const unsigned y = r % h.n[1], z = r / h.n[1];
            const int a = k - 5;
            // a thin axis has one face, both sides of the cell
            const int sh = h.n[a] > 1 ? (a == 0 ? 1 : (a == 1 ? nx : nxy)) : 0;
            const double *f = BF + (size_t)a * nface + (size_t)z * nxy + (size_t)y * nx + x;
            v = (f[0] + f[sh]) / 2;
        }
    } else {
        const size_t j = i - h.nu + h.bf0;
        const unsigned f = (unsigned)(j / 3);
        const int a = (int)(j - (size_t)f * 3);
        const int x = (int)(f % h.N[0]) - 2, y = (int)(f / h.N[0] % h.N[1]) - 2,
                  z = (int)(f / ((unsigned)h.N[0] * h.N[1])) - 2;
        if (x >= 0 && y >= 0 && z >= 0 && x < h.N[0] - 4 && y < h.N[1] - 4 && z < h.N[2] - 4)
            v = BF[(size_t)a * nface + (size_t)z * nxy + (size_t)y * nx + x];
    }
    out[t] = v;
}

// The reverse, into slot 0: cell-centred B and ghost faces are not stored.
__global__ void __launch_bounds__(kThreads) k_unpack(HostShape h, double *U, double *BF, size_t ncell,
                                                     size_t nface, size_t i0, size_t count,
                                                     const double *in) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const size_t i = i0 + t;
    if (i < h.nu) {
        const unsigned c = (unsigned)(i / h.nvar);
        const int k = (int)(i - (size_t)c * h.nvar);
        if (k < 5) U[(size_t)k * ncell + c] = in[t];
    } else {
        const size_t j = i - h.nu + h.bf0;
        const unsigned f = (unsigned)(j / 3);
        const int a = (int)(j - (size_t)f * 3);
        const int x = (int)(f % h.N[0]) - 2, y = (int)(f / h.N[0] % h.N[1]) - 2,
                  z = (int)(f / ((unsigned)h.N[0] * h.N[1])) - 2;
        if (x >= 0 && y >= 0 && z >= 0 && x < h.N[0] - 4 && y < h.N[1] - 4 && z < h.N[2] - 4)
            BF[(size_t)a * nface + ((size_t)z * (h.n[1] + 1) + y) * (h.n[0] + 1) + x] = in[t];
    }
}

// The time states into host memory, in stream order.
__global__ void __launch_bounds__(kThreads) k_report(const TimeState *ts, int ngrp, TimeState *out) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < ngrp) out[g] = ts[g];
}

}  // namespace kr
