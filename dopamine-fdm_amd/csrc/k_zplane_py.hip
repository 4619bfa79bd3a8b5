// k_zplane for a periodic y (FP64): z transforms and y FFT solve with each
// (kx, u) sub-plane held in registers: the plane is read and written once
// and passes through LDS for the exchanges of the z rows and twice for the y
// columns (half width), where the LDS-resident kernel (k_zfused.hip) takes
// every stage of every transform through LDS.  256x257x256: 171 us there (16
// modes a row), 96 here (32 modes a row, which shortens the x kernels).
// Bound by one workgroup a CU (two waves a SIMD) running its phases in turn.
#include <algorithm>

#include "k_zplane_impl.h"

namespace dfp {

// (N1, N2): rows of n modes; (NB, NCH): nym-1 = 8 NB NCH independent rows
#define DFP_ZPY_ROWS(X, ...) \
    X(2, 4, __VA_ARGS__) X(3, 4, __VA_ARGS__) X(2, 8, __VA_ARGS__) X(3, 8, __VA_ARGS__) X(4, 8, __VA_ARGS__) \
    X(6, 8, __VA_ARGS__) X(8, 8, __VA_ARGS__)
#define DFP_ZPY_COLS(X) X(1, 2) X(1, 4) X(1, 8) X(2, 8) X(2, 16)

// passes and chunks of nyp independent rows of n modes; false if the kernel does not take them
bool zplane_py_shape(int n, int nyp, size_t lds_limit, int& nb, int& nch) {
    bool rows = false;
#define DFP_ZPY_TRY(a, b, ...) rows = rows || a * b == n;
    DFP_ZPY_ROWS(DFP_ZPY_TRY, )
#undef DFP_ZPY_TRY
    nb = nch = 0;
#define DFP_ZPY_TRY(b, c) \
    if (8 * b * c == nyp) { nb = b; nch = c; }
    DFP_ZPY_COLS(DFP_ZPY_TRY)
#undef DFP_ZPY_TRY
    if (!rows || nb == 0 || n * nch > kZpyThreads) return false;
    return zplane_py_lds(std::max(n * nch, 64), n, nyp) <= lds_limit;
}

// rows of eight per chunk for every thread, kyy (twice, as the wall solve's two tables), w_n, w_nyp
size_t zplane_py_lds(int threads, int n, int nyp) {
    size_t slots = 0;
#define DFP_ZPY_PAD(a, b, ...) \
    if (a * b == n) slots = zplane_slots(a, b, 8, threads) + a * zplane_pad(a, b, 8);
    DFP_ZPY_ROWS(DFP_ZPY_PAD, )
#undef DFP_ZPY_PAD
    return sizeof(double2) * (slots + nyp) + 2 * sizeof(double) * (size_t)nyp;
}

hipError_t launch_zplane_py(dfp_plan* p, ZyPar<double2> zy) {
    const int n = p->fz.n, nyp = p->geo.nym - 1;
    zy.z.nch = p->zp_nch;
    zy.z.pp = std::max(1, 64 / (n * p->zp_nch));
    zy.z.nblocks = ceil_div(zy.z.nplanes, zy.z.pp);
    const int T = n * p->zp_nch * zy.z.pp, threads = ceil_div(T, 64) * 64;
    const size_t lds = zplane_py_lds(T, n, nyp);
    auto go = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(resident_grid(k, zy.z.nblocks, threads, lds)), dim3(threads), lds, p->stream, zy);
        return hipGetLastError();
    };
#define DFP_ZPY_GO(a, b, nb, nch) \
    if (a * b == n) return go(k_zplane_py<a, b, nb, nch>);
#define DFP_ZPY_CASE(nb, nch) \
    if (8 * nb * nch == nyp) { DFP_ZPY_ROWS(DFP_ZPY_GO, nb, nch) }
    DFP_ZPY_COLS(DFP_ZPY_CASE)
    return hipErrorInvalidValue;
}

}  // namespace dfp
