// The y solve of columns held in registers, chunks of L rows per thread.
//
// Every chunk runs the elimination b'(j) = b(j) - DL(j-1)/D'(j-1) b'(j-1)
// from a zero carry for its last row and for the product of its multipliers,
// the chunks' ends are chained through LDS (each thread folds the ends before
// its own), and the elimination proper runs from the chained carry: the same
// recurrence as one long sweep, with only the carries associated differently.
// The back substitution x(j) = (b'(j) - DU(j) x(j+1)) / D'(j) likewise from
// the top.  4 L + 2 nch serial steps in place of 2 nym.
#pragma once

#include "fft_lds.h"

namespace dfp {

// Keeps the compiler from carrying the FP64 image of an FP32 value from the
// first sweep over it into the second (twice the registers of the value).
__device__ __forceinline__ void keep_value(float2& v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }
__device__ __forceinline__ void keep_value(double2&) {}

// Where the chunks' ends lie in LDS: thread t's end value and multiplier
// product of the elimination (ce, cp) and of the back substitution (ge, gp).
struct FlatEnds {  // T threads, 48 T bytes
    double2* p;
    int T;
    __device__ __forceinline__ double2& ce(int t) const { return p[t]; }
    __device__ __forceinline__ double2& ge(int t) const { return p[T + t]; }
    __device__ __forceinline__ double& cp(int t) const { return reinterpret_cast<double*>(p + 2 * T)[t]; }
    __device__ __forceinline__ double& gp(int t) const { return reinterpret_cast<double*>(p + 2 * T)[T + t]; }
};
template <int W>
struct WaveEnds {  // each wave's in its own W bytes (3072 used)
    unsigned char* p;
    __device__ __forceinline__ unsigned char* at(int t, int size) const { return p + (t >> 6) * W + (t & 63) * size; }
    __device__ __forceinline__ double2& ce(int t) const { return *reinterpret_cast<double2*>(at(t, 16)); }
    __device__ __forceinline__ double2& ge(int t) const { return *reinterpret_cast<double2*>(at(t, 16) + 1024); }
    __device__ __forceinline__ double& cp(int t) const { return *reinterpret_cast<double*>(at(t, 8) + 2048); }
    __device__ __forceinline__ double& gp(int t) const { return *reinterpret_cast<double*>(at(t, 8) + 2560); }
};

// at(r): row j0 + r of this thread's column, r < L (C: double2, or float2,
// solved in FP64 and rounded where stored); rows past nym hold zero.
// pl[r] = 1/D'(j0 + r), plm = 1/D'(j0 - 1); dls[j] = DL(j-1), dus[j] = DU(j)
// for j < nch*L, zero outside the operator.  Thread t (act: one of the
// solving threads) owns chunk c of its column; the same column's next chunk is
// thread t + stride.  ends: LDS where thread t may write its own entries on
// entry, free again on return.  Every thread of the block must call it.
// zero: the column's solution is replaced by zero.
template <int L, typename C, typename At, typename Ends>
__device__ __forceinline__ void chunk_ysolve(At at, double (&pl)[L], double plm, const double* dls, const double* dus,
                                             int nym, int j0, int c, int nch, int stride, int t, bool act,
                                             bool zero, const Ends& ends) {
    using Rl = typename CplxT<C>::real;
    // elimination.  Rows past nym hold zero, take no multiplier and a zero
    // inverse pivot, so they carry nothing into the back substitution.
    if (j0 == 0) plm = 0.0;
    {
        double ex = 0.0, ey = 0.0, pi = 1.0, ip = plm;
#pragma unroll
        for (int r = 0; r < L; ++r) {
            if (j0 + r >= nym) pl[r] = 0.0;
            const double mu = dls[j0 + r] * ip;
            const C v = at(r);
            ex = (double)v.x - mu * ex;
            ey = (double)v.y - mu * ey;
            pi *= -mu;
            ip = pl[r];
        }
        if (act) {
            ends.ce(t) = make_double2(ex, ey);
            ends.cp(t) = pi;
        }
    }
    __syncthreads();
    {
        double bx = 0.0, by = 0.0, ip = plm;
#pragma unroll
        for (int r = 0; r < L; ++r) keep_value(at(r));
#pragma unroll 2
        for (int q = 0; q < c; ++q) {
            const double2 e = ends.ce(t - (c - q) * stride);
            const double f = ends.cp(t - (c - q) * stride);
            bx = e.x + f * bx;
            by = e.y + f * by;
        }
#pragma unroll
        for (int r = 0; r < L; ++r) {
            const double mu = dls[j0 + r] * ip;
            C& v = at(r);
            bx = (double)v.x - mu * bx;
            by = (double)v.y - mu * by;
            v = CplxT<C>::make((Rl)bx, (Rl)by);
            ip = pl[r];
        }
    }
    // back substitution, from the top
    {
        double gx = 0.0, gy = 0.0, pi = 1.0;
#pragma unroll
        for (int r = L - 1; r >= 0; --r) {
            const double d = dus[j0 + r];
            const C v = at(r);
            gx = ((double)v.x - d * gx) * pl[r];
            gy = ((double)v.y - d * gy) * pl[r];
            pi *= -d * pl[r];
        }
        if (act) {
            ends.ge(t) = make_double2(gx, gy);
            ends.gp(t) = pi;
        }
    }
    __syncthreads();
    {
        double xx = 0.0, xy = 0.0;
#pragma unroll
        for (int r = 0; r < L; ++r) keep_value(at(r));
#pragma unroll 2
        for (int q = nch - 1; q > c; --q) {
            const double2 e = ends.ge(t + (q - c) * stride);
            const double f = ends.gp(t + (q - c) * stride);
            xx = e.x + f * xx;
            xy = e.y + f * xy;
        }
#pragma unroll
        for (int r = L - 1; r >= 0; --r) {
            const double d = dus[j0 + r];
            C& v = at(r);
            xx = ((double)v.x - d * xx) * pl[r];
            xy = ((double)v.y - d * xy) * pl[r];
            v = CplxT<C>::make((Rl)xx, (Rl)xy);
        }
        if (zero) {
            asm volatile("");  // a branch, not a selection of every value
#pragma unroll
            for (int r = 0; r < L; ++r) at(r) = CplxT<C>::make((Rl)0, (Rl)0);
        }
    }
    __syncthreads();
}

}  // namespace dfp
