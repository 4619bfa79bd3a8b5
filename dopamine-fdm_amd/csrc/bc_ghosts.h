// The ghost copies of one interior value under apply_boundary_conditions
// (boundary_conditions.f90:186-260), for kernels that write the boundary
// conditions together with the field (a periodic x).
//
// The sequence x wrap, z wrap (or z walls), y walls (or y wrap), x wrap,
// z wrap leaves every ghost a function of one interior value: its x and z
// images (and, periodic, its y image) are copies, a wall row is the Robin
// expression of the row beside it with the slip length at the source's
// (i, k), a z wall plane is minus its neighbour (U, V) or zero (W), and a
// wall row of a z wall plane takes that plane's own slip length (no z wrap
// follows).  Kernels that write the field therefore write its images as well
// (scatter), or one launch fills every ghost row from its source (gather,
// k_ghost_rows in k_step.hip); nothing reads a ghost, so no order is needed
// between threads.  The arithmetic is the wall kernels' (k_step.hip), and the
// result is the sequence's bit for bit.
#pragma once

#include "dfp_internal.h"

namespace dfp {

// Robin wall data (boundary_conditions.f90:784-804) and the branch of each direction
struct BcArgs {
    const double* alpha[3];  // alpha_x (nx,2,nzg), alpha_y (nxg,2,nzg), alpha_z (nxg,2,nz)
    double dy1, dy2;         // y(2)-y(1), y(ny)-y(ny-1)
    double dg1, dg2;         // yg(2)-yg(1), yg(nyg)-yg(nyg-1)
    int ybc, zbc;
};

BcArgs make_bc(const dfp_plan* p, const double* ax, const double* ay, const double* az);
// every field has interior rows and planes, so each ghost has an interior source
inline bool bc_fusable(const Geo& g) { return g.xbc == 0 && g.ny > 2 && (g.zbc == 0 || g.nz > 2); }

// lower / upper wall row from the row beside it: y faces (V), y centres (U, W)
template <bool UPPER>
__device__ __forceinline__ double bc_robin(const BcArgs& b, int fi, double a, double v) {
#pragma clang fp contract(off)
    if (fi == 1) {
        const double d = UPPER ? b.dy2 : b.dy1;
        return a * v / d / (a / d + 1.0);
    }
    const double d = UPPER ? b.dg2 : b.dg1;
    return (2.0 * a / d - 1.0) * v / (2.0 * a / d + 1.0);
}

// (i, j, k) of field fi is itself a periodic image (the cells' duplicate of index 2)
__device__ __forceinline__ bool bc_image_x(int fi, int i, int n1) { return fi != 0 && i == n1 - 1; }
__device__ __forceinline__ bool bc_image_yz(const BcArgs& b, int fi, int j, int k, int n2, int n3) {
    return (b.ybc == 0 && fi != 1 && j == n2 - 1) || (b.zbc == 0 && fi != 2 && k == n3 - 1);
}
// row (j, k) has an image row: within two of the index 2 or n-1 that images copy
__device__ __forceinline__ bool bc_edge_yz(int j, int k, int n2, int n3) {
    return j <= 3 || j >= n2 - 2 || k <= 3 || k >= n3 - 2;
}

// x images of the values a, b at i, i+1 of one row (row[x], x = 1..n1)
__device__ __forceinline__ void bc_images_x(Glob<double>* row, int n1, int fi, int i, double a, double b, bool ok0,
                                            bool ok1) {
    if (fi == 0) {  // faces: nx <- 2, 1 <- nx-1
        if (ok0 && i == 2) row[n1] = a;
        if (ok1 && i + 1 == 2) row[n1] = b;
        if (ok0 && i == n1 - 1) row[1] = a;
        if (ok1 && i + 1 == n1 - 1) row[1] = b;
    } else {  // centres: nxg-1 <- 2, nxg <- 3, 1 <- nxg-2
        if (ok0 && (i == 2 || i == 3)) row[n1 - 3 + i] = a;
        if (ok1 && (i + 1 == 2 || i + 1 == 3)) row[n1 - 2 + i] = b;
        if (ok0 && i == n1 - 2) row[1] = a;
        if (ok1 && i + 1 == n1 - 2) row[1] = b;
    }
}

// Writes the image rows of the interior value v at (i, j, k) of field fi
// (extents n1, n2, n3; no image itself) with their own x images: every
// combination of a z and a y image but the row itself.  Only rows at an edge
// (bc_edge_yz) have any.  The loops stay rolled, for one value per thread: in
// the correction, whose threads hold 24, the same chain took 20 us unrolled
// (instruction fetches) and 33 us rolled at 16x16x16, against 3 us for the
// gather launch.
__device__ __forceinline__ void bc_images_yz(Glob<double>* F, int n1, int n2, int n3, int fi, int i, int j, int k,
                                             double v, const BcArgs& bc) {
#pragma unroll 1
    for (int zi = 0; zi < 4; ++zi) {
        int kk = zi == 0 ? k : 0, ka = k;  // destination plane, plane of the slip length
        double sg = 1.0;
        if (bc.zbc == 1) {
            if (zi == 1 && k == 2) kk = ka = 1;
            if (zi == 3 && k == n3 - 1) kk = ka = n3;
            if (zi != 0) sg = fi == 2 ? 0.0 : -1.0;
        } else if (fi == 2) {
            if (zi == 1 && k == 2) kk = n3;
            if (zi == 3 && k == n3 - 1) kk = 1;
        } else {
            if (zi == 1 && k == 2) kk = n3 - 1;
            if (zi == 2 && k == (n3 == 4 ? 2 : 3)) kk = n3;  // one independent plane: image of an image
            if (zi == 3 && k == n3 - 2) kk = 1;
        }
        if (kk == 0) continue;
        const double vz = sg == 1.0 ? v : (sg == 0.0 ? 0.0 : -v);
#pragma unroll 1
        for (int yi = 0; yi < 4; ++yi) {
            int jj = yi == 0 ? j : 0;
            double w = vz;
            if (bc.ybc == 1) {
                const auto al = gptr(bc.alpha[fi]) + (i - 1) + 2 * (long)(ka - 1) * n1;
                if (yi == 1 && j == 2) {
                    jj = 1;
                    w = bc_robin<false>(bc, fi, al[0], vz);
                }
                if (yi == 3 && j == n2 - 1) {
                    jj = n2;
                    w = bc_robin<true>(bc, fi, al[n1], vz);
                }
            } else if (fi == 1) {
                if (yi == 1 && j == 2) jj = n2;
                if (yi == 3 && j == n2 - 1) jj = 1;
            } else {
                if (yi == 1 && j == 2) jj = n2 - 1;
                if (yi == 2 && j == (n2 == 4 ? 2 : 3)) jj = n2;
                if (yi == 3 && j == n2 - 2) jj = 1;
            }
            if (jj == 0 || (jj == j && kk == k)) continue;
            const auto row = F + (long)(jj - 1) * n1 + (long)(kk - 1) * n1 * n2 - 1;
            row[i] = w;
            bc_images_x(row, n1, fi, i, w, 0.0, true, false);
        }
    }
}

}  // namespace dfp
