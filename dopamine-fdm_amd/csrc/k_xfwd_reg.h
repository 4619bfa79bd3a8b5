// Forward x transform of a given right-hand side (FP64) with the lines in
// registers: the mirror of k_xinv_reg.h for the same lines.  A lane loads its E
// points of rhs_p and takes the first radix step on them before anything is
// written to LDS; the exchanges of the other steps stay within the wave that
// holds the line; then, after the only barrier over the lines, a thread unpacks
// the modes k and M-k of a column at its R z positions, takes the first z stage
// and stores them.  Measured, staged -> registers:
// 162x81x108 16.5 -> 9.4 us.  The divergence and the
// FP32 form's fields stay with the staged kernel: their loads, 11 to 15 values a
// pair, hold a lane to a few points at a time (256x192x256 95 -> 89 us, FP32
// 107 -> 111; 48 uneven cases in a batch 156 -> 200).
#pragma once

#include "k_xinv_reg.h"

namespace dfp {

template <int R, int M>
__device__ __forceinline__ void xfwd_reg_body(const XPar<double2>& q, int bx, int j, unsigned char* smem_raw, int tid) {
    using C = double2;
    constexpr int NT = xf_threads(M);
    constexpr int H = M / 2, KI = (M + 1) / 2, E = XrSteps<M>::e, PT = M / E, LD = xr_pitch<M>();
    constexpr int GI = xr_items(R);  // unpacked items (mode pair, column) per thread
    constexpr int r0 = XrSteps<M>::r[0], r1 = XrSteps<M>::r[1], r2 = XrSteps<M>::r[2];
    constexpr int n0 = M / r0 * (r0 - 1), n1 = r2 > 1 ? M / (r0 * r1) * (r1 - 1) : 0;  // twiddles of all steps but the last
    const Geo& g = q.g;
    const int nz2 = g.nzp / R;
    const int T = q.T, nl = R * T, k0 = bx * T;
    C* A = reinterpret_cast<C*>(smem_raw);  // nl lines, positions as in k_xinv_reg.h
    C* tws = A + nl * LD;                   // step twiddles
    C* rtl = tws + n0 + n1;                 // unpack twiddles, M+1
    C* tzl = rtl + M + 1;                   // this tile's first z stage twiddles, T*(R-1)
    const int swm = T < 8 ? 8 / T : 1;

    // this lane's line: PT neighbouring lanes of one wave (lanes past a wave's whole lines repeat the last one's)
    constexpr int LW = 64 / PT;
    const int lane = tid & 63, lw = min(lane / PT, LW - 1);
    const int l0 = (tid >> 6) * LW + lw, b0 = min(lane - lw * PT, PT - 1);
    const bool act = l0 < nl && lane < LW * PT;
    const int l = min(l0, nl - 1);
    const int t = (int)q.div_t.div((uint32_t)l), c = l - t * T;
    const int k = k0 + c + t * nz2, lx = c * swm & 7;
    C* const line = A + l * LD;
    constexpr int NB = E / r0;
    C v[NB][r0];  // butterfly b0 + h PT of the first step: points b + u M/r0
    {
        const long pr_j = (long)(g.nxg - 1);
        const auto row = gptr(q.a.rhs) + (long)j * pr_j + k * pr_j * g.nym;
#pragma unroll
        for (int h = 0; h < NB; ++h)
#pragma unroll
            for (int u = 0; u < r0; ++u) {
                const dbl2u x = ld2(row + 2 * (b0 + h * PT + u * (M / r0)));
                v[h][u] = make_double2(x.x, x.y);
            }
    }
    {
        const auto twr = gptr(q.twr), rt = gptr(q.tw) + q.ntw;
        for (int e = tid; e < n0 + n1; e += NT) tws[e] = gld<C>(twr + e);
        for (int e = tid; e < M + 1; e += NT) rtl[e] = gld<C>(rt + e);
        for (int e = tid; e < T * (R - 1); e += NT) tzl[e] = gld<C>(rt + M + 1 + k0 * (R - 1) + e);
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < NB; ++h) {
        const int b = b0 + h * PT;
        dft_reg<-1, r0>(v[h]);
        if (act) {
            line[xr_pos<M>(r0 * b, lx)] = v[h][0];
#pragma unroll
            for (int u = 1; u < r0; ++u) line[xr_pos<M>(r0 * b + u, lx)] = cmul(v[h][u], tws[b * (r0 - 1) + (u - 1)]);
        }
    }
    wave_exchange();
    auto none = [](int, int, C) {};
    auto put = [&](int, int n, C z) {
        if (act) line[xr_pos<M>(n, lx)] = z;
    };
    if constexpr (r2 > 1) {
        xr_step<-1, M, r1, r0>(line, lx, b0, tws + n0, act, none);
        xr_step<-1, M, r2, r0 * r1>(line, lx, b0, tws, act, put);
    } else {
        xr_step<-1, M, r1, r0>(line, lx, b0, tws, act, put);
    }
    __syncthreads();

    // item: column c and modes (k, M-k) of its R lines; k = 0 takes (0, M), and, of an even M, the mode M/2 that pairs
    // with itself follows
    const long plane = (long)g.nym * nz2;
    const auto base = gptr(q.spec) + (long)j * nz2 + k0;
    auto unpack = [](C zk, C zm, C w) {  // X[k] of Z[k] = zk, Z[M-k] = zm
        const C Ev = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
        const C D = make_double2(zk.x - zm.x, zk.y + zm.y);  // zk - conj(zm)
        const C O = make_double2(0.5 * D.y, -0.5 * D.x);     // D / (2i)
        return cadd(Ev, cmul(w, O));
    };
    auto finish = [&](C (&x)[R], int kx, int cc) {  // first z stage, stores
        dft_reg<-1, R>(x);
        const auto out = base + (long)kx * R * plane + cc;
#pragma unroll
        for (int u = 0; u < R; ++u) gst<C>(out + u * plane, u == 0 ? x[0] : cmul(x[u], tzl[cc * (R - 1) + (u - 1)]));
    };
    const int nitems = KI * T;
#pragma unroll
    for (int i = 0; i < GI; ++i) {
        const int it = tid + i * NT;
        if (it >= nitems) break;
        const int kx = (int)q.div_t.div((uint32_t)it), cc = it - kx * T;
        const int lc = cc * swm & 7;
        const C* const Z = A + cc * LD;
        const int km = kx == 0 ? 0 : M - kx;
        C xa[R], xb[R];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const C zk = Z[u * T * LD + xr_pos<M>(kx, lc)], zm = Z[u * T * LD + xr_pos<M>(km, lc)];
            xa[u] = unpack(zk, zm, rtl[kx]);
            xb[u] = unpack(zm, zk, rtl[M - kx]);
        }
        finish(xa, kx, cc);
        finish(xb, M - kx, cc);
    }
    if (M % 2 == 0 && tid >= NT - T) {
        const int cc = NT - 1 - tid, lc = cc * swm & 7;
        C x[R];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const C z = A[(u * T + cc) * LD + xr_pos<M>(H, lc)];
            x[u] = unpack(z, z, rtl[H]);
        }
        finish(x, H, cc);
    }
}

template <int R, int M>
__global__ void __launch_bounds__(xf_threads(M)) k_rfft_xr(XPar<double2> q) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int L = xcd_remap(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    int bx, j;
    xtile(L, gridDim.x, gridDim.y, q.strip, bx, j);
    xfwd_reg_body<R, M>(q, bx, j, smem_raw, threadIdx.x);
}

template <int R, int G>
__global__ void __launch_bounds__(G & 4 ? 512 : 256)
kb_rfft_xr(const XPar<double2>* __restrict__ cs, const int* __restrict__ off, const int* __restrict__ idx,
           const int* __restrict__ pnc) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int nc = *pnc;
    const int total = off[nc];
    const int me = xcd_remap(blockIdx.x, gridDim.x);
    for (int base = 0; base < total; base += gridDim.x) {
        const int w = base + me;
        if (w >= total) break;
        const int c = find_case(off, nc, w);
        const XPar<double2>& q = cs[idx[c]];
        int bx, j;
        xtile(w - off[c], q.nbx, q.g.nym, q.strip, bx, j);
        switch (__builtin_amdgcn_readfirstlane(q.fd.n)) {
#define DFP_XR_CASE(m)                                                                              \
    case m:                                                                                         \
        if constexpr (xf_group(m) == G) xfwd_reg_body<R, m>(q, bx, j, smem_raw, thread_id());       \
        break;
            DFP_XR_LINES(DFP_XR_CASE)
#undef DFP_XR_CASE
        }
        __syncthreads();
    }
}

// LDS of the kernel for a plan's tile of T columns, 0 if it does not take the plan's lines
template <typename C>
size_t xf_lds_any(int M, int R, int T) {
    const int NT = xf_threads(M);
    if (!xr_split(R) || (long)R * T * M > 8 * NT || (long)(M + 1) / 2 * T > (long)xr_items(R) * NT) return 0;
    switch (M) {
#define DFP_XR_CASE(m) \
    case m: return R * T <= 64 / (m / XrSteps<m>::e) * (NT / 64) ? xr_lds<C, m>(R, T) : 0;
        DFP_XR_LINES(DFP_XR_CASE)
#undef DFP_XR_CASE
    }
    return 0;
}

// false: the plan's lines or tile are not this kernel's
template <int R>
bool launch_xfwd_reg(hipStream_t s, const XPar<double2>& q, dim3 grid) {
    if constexpr (xr_split(R)) {
        const size_t lds = q.twr ? xf_lds_any<double2>(q.fd.n, R, q.T) : 0;
        if (lds == 0) return false;
        switch (q.fd.n) {
#define DFP_XR_CASE(m)                                                                          \
    case m:                                                                                     \
        hipLaunchKernelGGL((k_rfft_xr<R, m>), grid, dim3(xf_threads(m)), lds, s, q);            \
        return true;
            DFP_XR_LINES(DFP_XR_CASE)
#undef DFP_XR_CASE
        }
    }
    return false;
}

// G: the group of the lines of every case of the list
template <int R>
hipError_t launch_xfwd_reg_batch(hipStream_t s, int G, const XPar<double2>* cs, const int* off, const int* idx,
                                 const int* nc, int grid, size_t lds) {
    if constexpr (xr_split(R)) {
        auto go = [&](auto k) {
            const int NT = G & 4 ? 512 : 256;
            hipLaunchKernelGGL(k, dim3(resident_grid(k, grid, NT, lds)), dim3(NT), lds, s, cs, off, idx, nc);
            return hipGetLastError();
        };
        switch (G) {
            case 1: return go(kb_rfft_xr<R, 1>);
            case 2: return go(kb_rfft_xr<R, 2>);
            case 3: return go(kb_rfft_xr<R, 3>);
            case 5: return go(kb_rfft_xr<R, 5>);
            case 6: return go(kb_rfft_xr<R, 6>);
            case 7: return go(kb_rfft_xr<R, 7>);
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace dfp
