// Inverse x transform with the lines in registers, for the lines of M = nxp/2
// packed points of DFP_XR_LINES (16 ... 256, 3-smooth).
//
// The staged kernel (xinv_body) takes every step through LDS: the gathered
// modes, the C2R packing and each radix-4 or -2 stage are a pass over the tile
// with a workgroup barrier on both sides, 12 accesses a point.  Here a thread
// gathers the modes k and M-k of its column at all R sub-lines, so it undoes
// the z split and packs Z[k] and Z[M-k] without an exchange; the lines are then
// transformed in two or three radix steps, E = 8 to 18 points a lane and PT = M/E
// neighbouring lanes a line (64/PT whole lines a wave), so each exchange stays
// within a wave and needs no barrier; the last step stores phi (and P) from
// registers.
// Six accesses a point and two barriers a tile.  Bound by HBM with P (303 MB at
// 256x192x256 in 62 us, 4.9 TB/s); measured, staged -> registers: 256x192x256
// 74 -> 62 us, FP32 46 -> 30 and (phi read) 86 -> 67, 512x384x512 486 -> 402,
// 256x257x256 86 -> 76, 64x64x64 7.5 -> 5.5.
//
// LDS position of point e of line l (column c of the tile): for M a multiple of
// 8, e ^ (e/8 mod 8) ^ lx(c), lx = c * (8/T) mod 8, which spreads the first step's
// strided writes, and the packing's writes of one mode in T neighbouring lines,
// over the banks (the reads run along the lines); for other M, e in lines of an
// odd pitch.
#pragma once

#include "fft_lds.h"

namespace dfp {

// z splits with a kernel, and the items (mode pair, column) that a thread gathers of a tile of up to 8 NT points
constexpr bool xr_split(int R) { return R <= 4 || R == 6 || R == 8 || R == 9; }
constexpr int xr_items(int R) { return (4 + R - 1) / R; }

// pitch of the lines in LDS, and position of point e in its line
template <int M>
constexpr int xr_pitch() { return M % 8 == 0 ? M : M | 1; }
template <int M>
__device__ __forceinline__ int xr_pos(int e, int lx) {
    if constexpr (M % 8 == 0) return e ^ (e >> 3 & 7) ^ lx;
    else return e;
}

// orders a wave's LDS accesses across the call, for exchanges among its lanes (which LDS serves in order)
__device__ __forceinline__ void wave_exchange() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// threadIdx.x for the bodies in a batched kernel, opaque to the compiler, so
// that each item forms what depends on it anew: held over the loop for every
// length, the LDS positions took up to 256 VGPRs and spilled
__device__ __forceinline__ int thread_id() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// One step of radix r and stride s on a line: this lane's 8/r butterflies.
// out(n, z) takes the results of the last step, the others stay in the line.
template <int SIGN, int M, int r, int s, typename C, typename Out>
__device__ __forceinline__ void xr_step(C* line, int lx, int b0, const C* tws, bool act, Out out) {
    constexpr int NB = XrSteps<M>::e / r, PT = M / XrSteps<M>::e;
    constexpr bool kLast = r * s == M;
    auto sw = [&](int e) { return xr_pos<M>(e, lx); };
    C v[NB][r];
#pragma unroll
    for (int h = 0; h < NB; ++h)
#pragma unroll
        for (int t = 0; t < r; ++t) v[h][t] = line[sw(b0 + h * PT + t * (M / r))];
    wave_exchange();
#pragma unroll
    for (int h = 0; h < NB; ++h) {
        const int b = b0 + h * PT;
        const int p = b / s, q = b - p * s;
        dft_reg<SIGN, r>(v[h]);
#pragma unroll
        for (int u = 0; u < r; ++u) {
            if constexpr (kLast) {
                out(h * r + u, q + s * u, v[h][u]);
            } else {
                const C z = u == 0 ? v[h][0] : twiddle<SIGN>(v[h][u], tws[p * (r - 1) + (u - 1)]);
                if (act) line[sw(q + s * (r * p + u))] = z;
            }
        }
    }
    wave_exchange();
}

// As xinv_body: last inverse z stage, C2R, phi (ACCUM: added to phi) with its
// duplicates and, with save_p, P = phi/(dt*c) with its ghosts.
template <typename C, int ACCUM, int R, int M>
__device__ __forceinline__ void xinv_reg_body(const XPar<C>& q, int bx, int j, unsigned char* smem_raw, double* wsum, int tid) {
    constexpr int NT = xr_threads<C>(M);
    constexpr int H = M / 2, KI = (M + 1) / 2, E = XrSteps<M>::e, PT = M / E, LD = xr_pitch<M>();
    constexpr int GI = xr_items(R);  // gathered items (mode pair, column) per thread
    constexpr int r0 = XrSteps<M>::r[0], r1 = XrSteps<M>::r[1], r2 = XrSteps<M>::r[2];
    constexpr int n0 = M / r0 * (r0 - 1), n1 = r2 > 1 ? M / (r0 * r1) * (r1 - 1) : 0;  // twiddles of all steps but the last
    const Geo& g = q.g;
    const int nz2 = g.nzp / R;
    const int T = q.T, nl = R * T, k0 = bx * T;
    C* A = reinterpret_cast<C*>(smem_raw);  // nl lines
    C* tws = A + nl * LD;                   // step twiddles
    C* rtl = tws + n0 + n1;                 // packing twiddles, M+1
    C* tzl = rtl + M + 1;                   // this tile's last z stage twiddles, T*(R-1)
    const int swm = T < 8 ? 8 / T : 1;

    // a periodic y's duplicate row nym-1 reads row 0 (projection.f90:350-354)
    const int js = (g.ybc == 0 && j == g.nym - 1) ? 0 : j;
    const int nitems = KI * T;
    const long plane = (long)g.nym * nz2;
    // item: column c and modes (k, M-k); k = 0 takes (0, M), and, of an even M, in xm the mode M/2 that pairs with itself
    C xa[GI][R], xb[GI][R], xm[R];
    const auto base = gptr(q.spec) + (long)js * nz2 + k0;
    if (M % 2 == 0 && tid < T) {
#pragma unroll
        for (int u = 0; u < R; ++u) xm[u] = gld<C>(base + ((long)H * R + u) * plane + tid);
    }
#pragma unroll
    for (int i = 0; i < GI; ++i) {
        const int it = min(tid + i * NT, nitems - 1);
        const int k = (int)q.div_t.div((uint32_t)it), c = it - k * T;
#pragma unroll
        for (int u = 0; u < R; ++u) {
            xa[i][u] = gld<C>(base + ((long)k * R + u) * plane + c);
            xb[i][u] = gld<C>(base + ((long)(M - k) * R + u) * plane + c);
        }
    }
    {
        const auto twr = gptr(q.twr), rt = gptr(q.tw) + q.ntw;
        for (int e = tid; e < n0 + n1; e += NT) tws[e] = gld<C>(twr + e);
        for (int e = tid; e < M + 1; e += NT) rtl[e] = gld<C>(rt + e);
        for (int e = tid; e < T * (R - 1); e += NT) tzl[e] = gld<C>(rt + M + 1 + k0 * (R - 1) + e);
    }
    __syncthreads();
    {
        // Z[k] of X[k] = x and X[M-k] = y
        auto pack = [](C x, C y, C w) {
            const C S = CplxT<C>::make(x.x + y.x, x.y - y.y);  // X[k] + conj X[M-k]
            const C D = CplxT<C>::make(x.x - y.x, x.y + y.y);  // X[k] - conj X[M-k]
            const C t = cmulc(D, w);
            return CplxT<C>::make(S.x - t.y, S.y + t.x);
        };
        auto undo_z = [&](C (&x)[R], int c) {
#pragma unroll
            for (int u = 1; u < R; ++u) x[u] = cmulc(x[u], tzl[c * (R - 1) + (u - 1)]);
            dft_reg<1, R>(x);
        };
#pragma unroll
        for (int i = 0; i < GI; ++i) {
            const int it = tid + i * NT;
            if (it < nitems) {
                const int k = (int)q.div_t.div((uint32_t)it), c = it - k * T;
                const int lx = c * swm & 7;
                auto sw = [&](int e) { return xr_pos<M>(e, lx); };
                undo_z(xa[i], c);
                undo_z(xb[i], c);
                const C wa = rtl[k], wb = rtl[M - k];
                C* const Z = A + c * LD;
#pragma unroll
                for (int t = 0; t < R; ++t) Z[t * T * LD + sw(k)] = pack(xa[i][t], xb[i][t], wa);
                if (k > 0) {
#pragma unroll
                    for (int t = 0; t < R; ++t) Z[t * T * LD + sw(M - k)] = pack(xb[i][t], xa[i][t], wb);
                }
            }
        }
        if (M % 2 == 0 && tid < T) {
            const int lx = tid * swm & 7;
            undo_z(xm, tid);
            const C w = rtl[H];
#pragma unroll
            for (int t = 0; t < R; ++t) A[(t * T + tid) * LD + xr_pos<M>(H, lx)] = pack(xm[t], xm[t], w);
        }
    }
    __syncthreads();

    // this lane's line: PT neighbouring lanes of one wave (lanes past a wave's whole lines repeat the last one's)
    constexpr int LW = 64 / PT;
    const int lane = tid & 63, lw = min(lane / PT, LW - 1);
    const int l0 = (tid >> 6) * LW + lw, b0 = min(lane - lw * PT, PT - 1);
    const bool act = l0 < nl && lane < LW * PT;
    const int l = min(l0, nl - 1);
    const int t = (int)q.div_t.div((uint32_t)l), c = l - t * T;
    const int k = k0 + c + t * nz2, lx = c * swm & 7;
    C* const line = A + l * LD;
    const long pr_j = (long)(g.nxg - 1), pr_k = pr_j * g.nym;
    const auto rr = gptr(q.rhs) + (long)j * pr_j + k * pr_k;
    double2 ph[E];
    int at[E];  // first x point of each pair
    auto none = [](int, int, C) {};
    auto take = [&](int o, int n, C z) {
        at[o] = 2 * n;
        ph[o] = make_double2((double)z.x * q.scale, (double)z.y * q.scale);
    };
    xr_step<1, M, r0, 1>(line, lx, b0, tws, act, none);
    if constexpr (r2 > 1) {
        xr_step<1, M, r1, r0>(line, lx, b0, tws + n0, act, none);
        xr_step<1, M, r2, r0 * r1>(line, lx, b0, tws, act, take);
    } else {
        xr_step<1, M, r1, r0>(line, lx, b0, tws, act, take);
    }

    double psum = 0.0;
    if (act) {
        if (q.pbar) {
            const double pb = gptr(q.pbar)[j];
#pragma unroll
            for (int o = 0; o < E; ++o) ph[o] = make_double2(ph[o].x + pb, ph[o].y + pb);
        }
        if constexpr (ACCUM != 0) {
            dbl2u old[E];
#pragma unroll
            for (int o = 0; o < E; ++o) old[o] = ld2(rr + at[o]);
#pragma unroll
            for (int o = 0; o < E; ++o) ph[o] = make_double2(ph[o].x + old[o].x, ph[o].y + old[o].y);
        }
        // rhs_p(i+2, j+2, k+2) and the duplicates (i = 0 -> nxp, k = 0 -> nzp; z walls have no z duplicate,
        // projection.f90:472-497)
        const bool zdup = k == 0 && g.zbc == 0;
#pragma unroll
        for (int o = 0; o < E; ++o) {
            psum += ph[o].x;
            psum += ph[o].y;
            st2(rr + at[o], ph[o].x, ph[o].y, true, true);
            if (at[o] == 0) rr[2 * M] = ph[o].x;
        }
        if (zdup) {
            const auto rz = rr + (long)g.nzp * pr_k;
#pragma unroll
            for (int o = 0; o < E; ++o) {
                st2(rz + at[o], ph[o].x, ph[o].y, true, true);
                if (at[o] == 0) rz[2 * M] = ph[o].x;
            }
        }
        if (q.save_p) {
            // every copy of these cells in P, as in xinv_body
#pragma unroll
            for (int o = 0; o < E; ++o) ph[o] = make_double2(ph[o].x / q.dtc, ph[o].y / q.dtc);
            const bool zw = g.zbc == 1;
            const int y1 = j == 0 ? 1 : 0, y2 = j == g.nym - 1 ? g.nyg : 0;
            const int z1 = zw ? (k == 0 ? 1 : 0) : (k == g.nzp - 1 ? 1 : 0);
            const int z2 = zw ? (k == g.nzp - 1 ? g.nzg : 0) : (k == 0 ? g.nzg - 1 : 0);
            const int z3 = zw ? 0 : (k == 1 % g.nzp ? g.nzg : 0);
            const auto P = gptr(q.P);
#pragma unroll 1
            for (int c3 = 0; c3 < 4; ++c3) {
                const int zz = c3 == 0 ? k + 2 : (c3 == 1 ? z1 : (c3 == 2 ? z2 : z3));
                if (zz == 0) continue;
#pragma unroll 1
                for (int b = 0; b < 3; ++b) {
                    const int yy = b == 0 ? j + 2 : (b == 1 ? y1 : y2);
                    if (yy == 0) continue;
                    const auto Pr = P + (long)(yy - 1) * g.nxg + (long)(zz - 1) * g.nxg * g.nyg;
#pragma unroll
                    for (int o = 0; o < E; ++o) {
                        st2(Pr + at[o] + 1, ph[o].x, ph[o].y, true, true);  // x = i+2, i+3
                        if (at[o] == 0) {
                            Pr[g.nxg - 2] = ph[o].x;  // x = nxg-1
                            Pr[g.nxg - 1] = ph[o].y;  // x = nxg
                        }
                        if (at[o] == 2 * M - 2) Pr[0] = ph[o].y;  // x = 1
                    }
                }
            }
        }
    }
    if (q.part0 && j == 0) {
        const double sblk = block_sum<NT>(psum, wsum);
        if (tid == 0) gptr(q.part0)[bx] = sblk;
    }
}

// LDS of the kernel for nl = R*T lines
template <typename C, int M>
constexpr size_t xr_lds(int R, int T) {
    constexpr int r0 = XrSteps<M>::r[0], r1 = XrSteps<M>::r[1], r2 = XrSteps<M>::r[2];
    return sizeof(C) * ((size_t)R * T * xr_pitch<M>() + M / r0 * (r0 - 1) + (r2 > 1 ? M / (r0 * r1) * (r1 - 1) : 0) + M + 1 +
                        (size_t)T * (R - 1));
}

template <typename C, int ACCUM, int R, int M>
__global__ void __launch_bounds__(xr_threads<C>(M)) k_irfft_xr(XPar<C> q) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int L = xcd_remap(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    int bx, j;
    xtile(L, gridDim.x, gridDim.y, q.strip, bx, j);
    __shared__ double wsum[xr_threads<C>(M) / 64];
    xinv_reg_body<C, ACCUM, R, M>(q, bx, j, smem_raw, wsum, threadIdx.x);
}

// one workgroup per work item, or persistent, as the other batched kernels; G: the group of its cases' lines
template <typename C, int ACCUM, int R, int G>
__global__ void __launch_bounds__(G & 4 ? 512 : 256)
kb_irfft_xr(const XPar<C>* __restrict__ cs, const int* __restrict__ off, const int* __restrict__ idx,
            const int* __restrict__ pnc) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double wsum[8];
    const int nc = *pnc;
    const int total = off[nc];
    const int me = xcd_remap(blockIdx.x, gridDim.x);
    for (int base = 0; base < total; base += gridDim.x) {
        const int w = base + me;
        if (w >= total) break;
        const int c = find_case(off, nc, w);
        const XPar<C>& q = cs[idx[c]];
        int bx, j;
        xtile(w - off[c], q.nbx, q.g.nym, q.strip, bx, j);
        switch (__builtin_amdgcn_readfirstlane(q.fd.n)) {
#define DFP_XR_CASE(m)                                                                                              \
    case m:                                                                                                         \
        if constexpr (xr_group<C>(m) == G) xinv_reg_body<C, ACCUM, R, m>(q, bx, j, smem_raw, wsum, thread_id());    \
        break;
            DFP_XR_LINES(DFP_XR_CASE)
#undef DFP_XR_CASE
        }
        __syncthreads();
    }
}

// LDS of the kernel for a plan's tile of T columns, 0 if it does not take the plan's lines
template <typename C>
size_t xr_lds_any(int M, int R, int T) {
    if (!xr_split(R)) return 0;
    if ((long)R * T * M > 8 * xr_threads<C>(M)) return 0;
    // the items of the gather, and the lines of the waves
    if ((long)(M + 1) / 2 * T > (long)xr_items(R) * xr_threads<C>(M)) return 0;
    switch (M) {
#define DFP_XR_CASE(m)                                                                                       \
    case m:                                                                                                  \
        return R * T <= 64 / (m / XrSteps<m>::e) * (xr_threads<C>(m) / 64) ? xr_lds<C, m>(R, T) : 0;
        DFP_XR_LINES(DFP_XR_CASE)
#undef DFP_XR_CASE
    }
    return 0;
}

// G: the group of the lines of every case of the list
template <typename C, int ACCUM, int R>
hipError_t launch_xinv_reg_batch(hipStream_t s, int G, const XPar<C>* cs, const int* off, const int* idx,
                                 const int* nc, int grid, size_t lds) {
    if constexpr (xr_split(R)) {
        auto go = [&](auto k) {
            const int NT = G & 4 ? 512 : 256;
            hipLaunchKernelGGL(k, dim3(resident_grid(k, grid, NT, lds)), dim3(NT), lds, s, cs, off, idx, nc);
            return hipGetLastError();
        };
        switch (G) {
            case 1: return go(kb_irfft_xr<C, ACCUM, R, 1>);
            case 2: return go(kb_irfft_xr<C, ACCUM, R, 2>);
            case 3: return go(kb_irfft_xr<C, ACCUM, R, 3>);
            case 5: return go(kb_irfft_xr<C, ACCUM, R, 5>);
        }
        if constexpr (sizeof(C) == sizeof(float2)) {  // FP64: 512 threads for 256 points only
            if (G == 6) return go(kb_irfft_xr<C, ACCUM, R, 6>);
            if (G == 7) return go(kb_irfft_xr<C, ACCUM, R, 7>);
        }
    }
    return hipErrorInvalidValue;
}

// false: the plan's lines or tile are not this kernel's
template <typename C, int ACCUM, int R>
bool launch_xinv_reg(hipStream_t s, const XPar<C>& q, dim3 grid) {
    if constexpr (xr_split(R)) {
        if (!q.twr || xr_lds_any<C>(q.fd.n, R, q.T) == 0) return false;
        auto go = [&](auto m) {
            constexpr int M = decltype(m)::value;
            constexpr int NT = xr_threads<C>(M);
            hipLaunchKernelGGL((k_irfft_xr<C, ACCUM, R, M>), grid, dim3(NT), (xr_lds<C, M>(R, q.T)), s, q);
            return true;
        };
        switch (q.fd.n) {
#define DFP_XR_CASE(m) \
    case m: return go(std::integral_constant<int, m>{});
            DFP_XR_LINES(DFP_XR_CASE)
#undef DFP_XR_CASE
        }
    }
    return false;
}

}  // namespace dfp
