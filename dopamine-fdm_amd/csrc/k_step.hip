// The step either side of the projection for a periodic x (the channel, the
// periodic box, the duct), one rank, on device-resident fields:
//   k_rk_update     RK3 stage update of the interior  time_integration.f90:256-258,
//                                                     :394-396, :526-531
//   k_wrap_x/z      periodic ghost planes             boundary_conditions.f90:263-289,
//                                                     :580-602
//   k_robin_y       Robin (slip-length) wall rows     boundary_conditions.f90:784-804
//   k_wrap_y        periodic y ghost rows (y_bc_type = 0, the periodic box)
//                                                     boundary_conditions.f90:762-781
//   k_wall_z        z wall planes (the duct)          boundary_conditions.f90:737-758
// apply_boundary_conditions (:186-260) is the sequence x wrap, z wrap (or
// z walls, :215-223), y walls (or y wrap, :229-233), x wrap, z wrap (none
// with z walls); on one rank its halo exchanges (:170-183) exchange nothing.  Each launch covers the three fields (blockIdx.z); arithmetic is
// kept operation for operation (no contraction), so results equal the CPU
// path bit for bit.
// A substage does not launch that sequence: k_rk_update and k_correct
// (k_stencil.hip) write the ghosts with the field (bc_ghosts.h).
#include <algorithm>

#include "bc_ghosts.h"

namespace dfp {

// extents of U (0), V (1), W (2)
struct Field3 {
    double* F[3];
    int n1[3], n2[3], n3[3];
};

static Field3 field3(const Geo& g, double* U, double* V, double* W) {
    Field3 f{};
    f.F[0] = U; f.F[1] = V; f.F[2] = W;
    f.n1[0] = g.nx;  f.n2[0] = g.nyg; f.n3[0] = g.nzg;
    f.n1[1] = g.nxg; f.n2[1] = g.ny;  f.n3[1] = g.nzg;
    f.n1[2] = g.nxg; f.n2[2] = g.nyg; f.n3[2] = g.nz;
    return f;
}

struct RkArgs {
    const double* Fo[3];      // Uo, Vo, Wo
    const double* R[3][3];    // [field][stage term]: interior-shaped right-hand sides
    double c[3];              // rk_coef(stage, 1:stage)
    double dt;
};

// one thread per interior element (i, j) of plane k = blockIdx.y + 2 of field
// blockIdx.z.  BC: the images of every element are written too (the boundary
// conditions that follow the update in a substage), and elements that are
// images themselves are left to their sources.  Bound by HBM (five streams at
// stage 3: 1.5 GB in 300 us at 256x192x256, 5.0 TB/s, with or without the
// images; 2.7 us without and 4.9 us with them at 16x16x16, where a launch for
// them would take 3 us and its gap).
template <int STAGE, bool BC>
__global__ void __launch_bounds__(256) k_rk_update(Field3 f, RkArgs a, BcArgs bc) {
#pragma clang fp contract(off)
    const int fi = blockIdx.z;
    const int n1 = f.n1[fi], n2 = f.n2[fi], n3 = f.n3[fi];
    const int ni = n1 - 2, nj = n2 - 2;
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int k = 2 + blockIdx.y;
    if (t >= ni * nj || k > n3 - 1) return;
    const int jj = t / ni, ii = t - jj * ni;
    if (BC && (bc_image_x(fi, ii + 2, n1) || bc_image_yz(bc, fi, jj + 2, k, n2, n3))) return;
    const long e = (ii + 1) + (long)(jj + 1) * n1 + (long)(k - 1) * n1 * n2;  // (i, j, k) = (ii+2, jj+2, k)
    const long r = ii + (long)jj * ni + (long)(k - 2) * ni * nj;             // interior array
    const double fo = a.Fo[fi][e];
    double v;
    if (STAGE == 1) {
        v = fo + a.dt * a.c[0] * a.R[fi][0][r];
    } else if (STAGE == 2) {
        v = fo + a.dt * (a.c[0] * a.R[fi][0][r] + a.c[1] * a.R[fi][1][r]);
    } else {
        v = fo + a.dt * (a.c[0] * a.R[fi][0][r] + a.c[1] * a.R[fi][1][r] + a.c[2] * a.R[fi][2][r]);
    }
    f.F[fi][e] = v;
    if (BC) {
        bc_images_x(gptr(f.F[fi]) + (e - ii - 2), n1, fi, ii + 2, v, 0.0, true, false);
        if (bc_edge_yz(jj + 2, k, n2, n3))
            bc_images_yz(gptr(f.F[fi]), n1, n2, n3, fi, ii + 2, jj + 2, k, v, bc);
    }
}

// x ghost planes over (j, k): U faces (1 <- nx-1, nx <- 2), V and W centres
// (1 <- nxg-2, nxg-1 <- 2, nxg <- 3)
__global__ void __launch_bounds__(256) k_wrap_x(Field3 f) {
    const int fi = blockIdx.z;
    const int n1 = f.n1[fi], n2 = f.n2[fi], n3 = f.n3[fi];
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long)n2 * n3) return;
    double* row = f.F[fi] + t * n1;  // F(:, j, k)
    // in the reference's statement order, like the z wraps (with nxp >= 2 no
    // copy reads a plane an earlier one wrote)
    if (fi == 0) {
        row[0] = row[n1 - 2];
        row[n1 - 1] = row[1];
    } else {
        row[0] = row[n1 - 3];
        row[n1 - 2] = row[1];
        row[n1 - 1] = row[2];
    }
}

// z ghost planes over (i, j): U and V centres (1 <- nzg-2, nzg-1 <- 2,
// nzg <- 3), W faces (1 <- nz-1, nz <- 2)
__global__ void __launch_bounds__(256) k_wrap_z(Field3 f) {
    const int fi = blockIdx.z;
    const int n1 = f.n1[fi], n2 = f.n2[fi], n3 = f.n3[fi];
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long pl = (long)n1 * n2;
    if (t >= pl) return;
    double* F = f.F[fi] + t;  // F(i, j, :) with stride pl
    // in the reference's statement order (with nzp = 1, nzg-1 = 3 is read
    // after it is written)
    if (fi == 2) {
        F[0] = F[(n3 - 2) * pl];
        F[(n3 - 1) * pl] = F[pl];
    } else {
        F[0] = F[(n3 - 3) * pl];
        F[(n3 - 2) * pl] = F[pl];
        F[(n3 - 1) * pl] = F[2 * pl];
    }
}

// y ghost rows over (i, k): V faces (1 <- ny-1, ny <- 2), U and W centres
// (1 <- nyg-2, nyg-1 <- 2, nyg <- 3), in the reference's statement order
__global__ void __launch_bounds__(256) k_wrap_y(Field3 f) {
    const int fi = blockIdx.z;
    const int n1 = f.n1[fi], n2 = f.n2[fi], n3 = f.n3[fi];
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long)n1 * n3) return;
    const long k = t / n1, i = t - k * n1;
    double* F = f.F[fi] + i + k * (long)n1 * n2;  // F(i, 1, k), stride n1 in y
    if (fi == 1) {
        F[0] = F[(long)(n2 - 2) * n1];
        F[(long)(n2 - 1) * n1] = F[n1];
    } else {
        F[0] = F[(long)(n2 - 3) * n1];
        F[(long)(n2 - 2) * n1] = F[n1];
        F[(long)(n2 - 1) * n1] = F[2 * (long)n1];
    }
}

// z wall planes over (i, j): W faces no-penetration (1 and nz zero), U and
// V centres no-slip by mirroring (1 <- -2, nzg <- -(nzg-1))
__global__ void __launch_bounds__(256) k_wall_z(Field3 f) {
    const int fi = blockIdx.z;
    const int n1 = f.n1[fi], n2 = f.n2[fi], n3 = f.n3[fi];
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long pl = (long)n1 * n2;
    if (t >= pl) return;
    double* F = f.F[fi] + t;  // F(i, j, :) with stride pl
    if (fi == 2) {
        F[0] = 0.0;
        F[(n3 - 1) * pl] = 0.0;
    } else {
        F[0] = -F[pl];
        F[(n3 - 1) * pl] = -F[(n3 - 2) * pl];
    }
}

// wall rows over (i, k): V faces (id 1), U and W centres (id 2)
__global__ void __launch_bounds__(256) k_robin_y(Field3 f, BcArgs a) {
    const int fi = blockIdx.z;
    const int n1 = f.n1[fi], n2 = f.n2[fi], n3 = f.n3[fi];
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long)n1 * n3) return;
    const long k = t / n1, i = t - k * n1;
    double* F = f.F[fi] + i + k * (long)n1 * n2;  // F(i, 1, k), stride n1 in y
    const double a1 = a.alpha[fi][i + 2 * k * (long)n1];
    const double a2 = a.alpha[fi][i + n1 + 2 * k * (long)n1];
    // lower wall first, then the upper one, which reads row n2-1 after the
    // lower row is written (they coincide for V with one cell between the walls)
    F[0] = bc_robin<false>(a, fi, a1, F[n1]);
    F[(long)(n2 - 1) * n1] = bc_robin<true>(a, fi, a2, F[(long)(n2 - 2) * n1]);
}

// Ghost rows of one field (blockIdx.z), each element from its interior source
// (bc_ghosts.h): the z ghost planes, the y ghost rows of the planes between
// them, and, with x_part, the x ghosts of every row left.  One launch in place
// of the sequence of five (39 us at 256x192x256, 13 us at 16x16x16).  x_part is
// left out after the correction, which writes its x images itself: the rows
// alone take 8.8 us at 256x192x256 and 3 us at 16x16x16, bound by latency.
__global__ void __launch_bounds__(256) k_ghost_rows(Field3 f, BcArgs bc, int x_part) {
    const int fi = blockIdx.z;
    const int n1 = f.n1[fi], n2 = f.n2[fi], n3 = f.n3[fi];
    // ghosts per direction: indices 1 and n, and n-1 where it duplicates index 2
    const bool dx = fi != 0, dy = bc.ybc == 0 && fi != 1, dz = bc.zbc == 0 && fi != 2;
    const int gx = dx ? 3 : 2, gy = dy ? 3 : 2, gz = dz ? 3 : 2;
    const int nj = n2 - gy, nk = n3 - gz;  // rows, planes that are no ghosts: 2 .. nj+1, 2 .. nk+1
    const long rows = (long)gz * n2 + (long)gy * nk;
    long t = (long)blockIdx.x * 256 + threadIdx.x;
    int i, j, k;
    if (t < rows * n1) {
        const int r = (int)(t / n1);
        i = 1 + (int)(t - (long)r * n1);
        if (r < gz * n2) {
            const int q = r / n2;
            j = 1 + r - q * n2;
            k = q == 0 ? 1 : n3 - q + 1;
        } else {
            const int s = r - gz * n2, q = s / nk;
            k = 2 + s - q * nk;
            j = q == 0 ? 1 : n2 - q + 1;
        }
    } else {
        t -= rows * n1;
        if (!x_part || t >= (long)gx * nj * nk) return;
        const int r = (int)(t / gx), q = (int)(t - (long)r * gx);
        i = q == 0 ? 1 : n1 - q + 1;
        k = 2 + r / nj;
        j = 2 + r - (k - 2) * nj;
    }
    // source of a periodic index: 1 <- the last independent one, n-1 (duplicated) <- 2, n <- the one after
    auto source = [](int e, int n, bool dup) {
        if (e == 1) return dup ? n - 2 : n - 1;
        if (!dup) return e == n ? 2 : e;
        if (e == n) return n == 4 ? 2 : 3;  // one independent index: image of an image
        return e == n - 1 ? 2 : e;
    };
    const int si = source(i, n1, dx);
    int sj = j, sk = k, ka = k;
    double sign = 1.0;
    if (bc.zbc == 0) {
        sk = ka = source(k, n3, dz);
    } else if (k == 1 || k == n3) {
        sk = k == 1 ? 2 : n3 - 1;
        sign = fi == 2 ? 0.0 : -1.0;
    }
    if (bc.ybc == 0) sj = source(j, n2, dy);
    else sj = j == 1 ? 2 : (j == n2 ? n2 - 1 : j);
    const auto F = gptr(f.F[fi]);
    const double s = F[(si - 1) + (long)(sj - 1) * n1 + (long)(sk - 1) * n1 * n2];
    double v = sign == 1.0 ? s : (sign == 0.0 ? 0.0 : -s);
    if (bc.ybc == 1 && sj != j) {
        const auto al = gptr(bc.alpha[fi]) + (si - 1) + 2 * (long)(ka - 1) * n1;
        v = j == 1 ? bc_robin<false>(bc, fi, al[0], v) : bc_robin<true>(bc, fi, al[n1], v);
    }
    F[(i - 1) + (long)(j - 1) * n1 + (long)(k - 1) * n1 * n2] = v;
}

BcArgs make_bc(const dfp_plan* p, const double* ax, const double* ay, const double* az) {
    BcArgs r{};
    r.alpha[0] = ax; r.alpha[1] = ay; r.alpha[2] = az;
    const auto& y = p->hy;
    const auto& yg = p->hyg;
    r.dy1 = y[1] - y[0];
    r.dy2 = y[y.size() - 1] - y[y.size() - 2];
    r.dg1 = yg[1] - yg[0];
    r.dg2 = yg[yg.size() - 1] - yg[yg.size() - 2];
    r.ybc = p->geo.ybc;
    r.zbc = p->geo.zbc;
    return r;
}

hipError_t launch_rk_update(dfp_plan* p, int stage, double* U, double* V, double* W, const double* const Fo[3],
                            const double* const* R[3], const double* c, double dt, const BcArgs* bc) {
    const Field3 f = field3(p->geo, U, V, W);
    RkArgs a{};
    for (int fi = 0; fi < 3; ++fi) {
        a.Fo[fi] = Fo[fi];
        for (int s = 0; s < stage; ++s) a.R[fi][s] = R[fi][s];
    }
    for (int s = 0; s < stage; ++s) a.c[s] = c[s];
    a.dt = dt;
    long plane = 0;
    for (int fi = 0; fi < 3; ++fi) plane = std::max(plane, (long)(f.n1[fi] - 2) * (f.n2[fi] - 2));
    int n3 = 0;
    for (int fi = 0; fi < 3; ++fi) n3 = std::max(n3, f.n3[fi] - 2);
    const dim3 grid(ceil_div(plane, 256), n3, 3);
    const int slot = prof_begin(p, "rk_update");
    auto go = [&](auto k) { hipLaunchKernelGGL(k, grid, dim3(256), 0, p->stream, f, a, bc ? *bc : BcArgs{}); };
    if (bc) {
        if (stage == 1) go(k_rk_update<1, true>);
        else if (stage == 2) go(k_rk_update<2, true>);
        else go(k_rk_update<3, true>);
    } else {
        if (stage == 1) go(k_rk_update<1, false>);
        else if (stage == 2) go(k_rk_update<2, false>);
        else go(k_rk_update<3, false>);
    }
    prof_end(p, slot);
    return hipGetLastError();
}

static void launch_ghost_rows(dfp_plan* p, const Field3& f, const BcArgs& bc, int x_part) {
    long n = 0;
    for (int fi = 0; fi < 3; ++fi) {
        const long gy = bc.ybc == 0 && fi != 1 ? 3 : 2, gz = bc.zbc == 0 && fi != 2 ? 3 : 2, gx = fi != 0 ? 3 : 2;
        const long nj = f.n2[fi] - gy, nk = f.n3[fi] - gz;
        n = std::max(n, (gz * f.n2[fi] + gy * nk) * f.n1[fi] + (x_part ? gx * nj * nk : 0));
    }
    hipLaunchKernelGGL(k_ghost_rows, dim3(ceil_div(n, 256), 1, 3), dim3(256), 0, p->stream, f, bc, x_part);
}

hipError_t launch_ghost_yz(dfp_plan* p, double* U, double* V, double* W, const BcArgs& bc) {
    const int slot = prof_begin(p, "apply_bc");
    launch_ghost_rows(p, field3(p->geo, U, V, W), bc, 0);
    prof_end(p, slot);
    return hipGetLastError();
}

// the sequence of boundary_conditions.f90:186-260, or one gather launch where
// every ghost has an interior source
hipError_t launch_apply_bc(dfp_plan* p, double* U, double* V, double* W, const double* ax, const double* ay,
                           const double* az) {
    const Field3 f = field3(p->geo, U, V, W);
    const BcArgs r = make_bc(p, ax, ay, az);
    long px = 0, pz = 0, py = 0;
    for (int fi = 0; fi < 3; ++fi) {
        px = std::max(px, (long)f.n2[fi] * f.n3[fi]);
        pz = std::max(pz, (long)f.n1[fi] * f.n2[fi]);
        py = std::max(py, (long)f.n1[fi] * f.n3[fi]);
    }
    const int slot = prof_begin(p, "apply_bc");
    if (bc_fusable(p->geo)) {
        launch_ghost_rows(p, f, r, 1);
        prof_end(p, slot);
        return hipGetLastError();
    }
    for (int pass = 0; pass < 2; ++pass) {
        hipLaunchKernelGGL(k_wrap_x, dim3(ceil_div(px, 256), 1, 3), dim3(256), 0, p->stream, f);
        if (p->geo.zbc == 0)
            hipLaunchKernelGGL(k_wrap_z, dim3(ceil_div(pz, 256), 1, 3), dim3(256), 0, p->stream, f);
        else if (pass == 0)
            hipLaunchKernelGGL(k_wall_z, dim3(ceil_div(pz, 256), 1, 3), dim3(256), 0, p->stream, f);
        if (pass == 0 && p->geo.ybc == 0)
            hipLaunchKernelGGL(k_wrap_y, dim3(ceil_div(py, 256), 1, 3), dim3(256), 0, p->stream, f);
        else if (pass == 0)
            hipLaunchKernelGGL(k_robin_y, dim3(ceil_div(py, 256), 1, 3), dim3(256), 0, p->stream, f, r);
    }
    prof_end(p, slot);
    return hipGetLastError();
}

}  // namespace dfp
