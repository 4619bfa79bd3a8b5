// Dispatch of the register-plane z kernels (k_zplane_impl.h).
#include "k_zplane_impl.h"

namespace dfp {

#define DFP_ZP_EXT(a, b, r)           \
    DFP_ZP_EXTERN(double2, a, b, r)   \
    DFP_ZP_EXTERN(float2, a, b, r)
DFP_ZP_SHORT(DFP_ZP_EXT)
DFP_ZP_LONG(DFP_ZP_EXT)

template <typename C>
hipError_t launch_zplane(dfp_plan* p, const ZPar<C>& zp) {
    const bool f32 = sizeof(C) == sizeof(float2);
    const size_t lds = z_lds_bytes(p, f32);
    const int threads = ceil_div((long)p->fz.n * zp.nch * zp.pp, 64) * 64;
    const int slot = prof_begin(p, f32 ? "zsolve32" : "zsolve");
    hipError_t e = hipErrorInvalidValue;
    switch (p->fz.n) {
#define DFP_ZP_CASE(a, b, r)                                                             \
    case a * b:                                                                          \
        e = launch_zplane_n<C, a, b, r>(p->stream, p->zp_nb, zp, threads, lds);          \
        break;
        DFP_ZP_SHORT(DFP_ZP_CASE)
        DFP_ZP_LONG(DFP_ZP_CASE)
#undef DFP_ZP_CASE
    }
    prof_end(p, slot);
    return e;
}
template hipError_t launch_zplane<double2>(dfp_plan*, const ZPar<double2>&);
template hipError_t launch_zplane<float2>(dfp_plan*, const ZPar<float2>&);

template <typename C>
hipError_t launch_zplane_batch(hipStream_t s, int variant, const ZPar<C>* cs, const int* off, const int* idx,
                               const int* nc, int grid, size_t lds, int wide) {
    const int nb = (variant - kZvPlane) / 1024, n1 = (variant & 1023) / 32, n2 = variant & 31;
    const int threads = wide ? zplane_threads(n1 * n2, nb) : kZpBatchThreads;
    switch (n1 * n2) {
#define DFP_ZP_CASE(a, b, r) \
    case a * b: return launch_zplane_batch_n<C, a, b, r>(s, nb, cs, off, idx, nc, grid, threads, lds);
        DFP_ZP_SHORT(DFP_ZP_CASE)
        DFP_ZP_LONG(DFP_ZP_CASE)
#undef DFP_ZP_CASE
    }
    return hipErrorInvalidValue;
}
template hipError_t launch_zplane_batch<double2>(hipStream_t, int, const ZPar<double2>*, const int*, const int*,
                                                 const int*, int, size_t, int);
template hipError_t launch_zplane_batch<float2>(hipStream_t, int, const ZPar<float2>*, const int*, const int*,
                                                const int*, int, size_t, int);

}  // namespace dfp
