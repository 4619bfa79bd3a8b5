// z transforms and y solve of one (kx, u) sub-plane held in registers: the
// rows are read once and written once (32 H bytes in FP64, 16 H in the FP32
// form, and the pivots), where the streaming kernel (k_zsolve.hip) writes the
// eliminated rows back and reads them again.
//
// A plane of nym rows of n = N1*N2 modes is cut into nch chunks of L = BR*NB
// consecutive rows.  A workgroup has n*nch threads per plane (and PP planes,
// where one plane would leave a wavefront empty); thread (chunk c, mode m)
// owns rows cL .. cL+L-1 of mode m.
//
//   forward z transform, BR rows of every chunk at a time (NB passes): each
//   thread loads BR/N2 items (row, i1) of N2 points straight from HBM,
//   transforms them in registers, exchanges through LDS for the length-N1
//   step (the two-step transform and LDS layout of k_zsolve.hip), and takes
//   its BR rows of its mode back into registers: through LDS again, or, for
//   16, 32 and 64 modes, across the lanes of its wave;
//   y solve in chunks (ychunk.h), with the plan's inverse pivots in registers;
//   inverse z transform: the same steps backwards, stored from registers.
//
// Bound by HBM for the rows' loads and stores, in which all workgroups are at
// first in step, with the transforms and the solve between (9 us a plane of
// 192 x 64 modes, 12 with its stores; 129 x 4 such planes on 256 CUs leave a
// third round of four).  With the exchanges free of barriers and of address
// arithmetic (kLane below): 256x192x256 73 -> 64 us, inflow (1024 planes)
// 100 -> 88 us = 4.6 TB/s, periodic y 256x257x256 105 -> 96 us.
//
// All of a plane's loads are in flight at once and no wave waits for another's
// sweep: the serial part is 4 L + 2 nch steps instead of 2 nym.  The working
// set (L complex values and L pivots per thread) is what limits it: planes
// that need more threads than zplane_threads stay with the streaming kernel.
#pragma once

#include "ychunk.h"

namespace dfp {

// Exchanges the register index r = 0..7 of v with bits 3..5 of the lane:
// v[r] of lane (h, k) becomes v[h] of lane (r, k), k = lane % 8.  One register
// bit and one lane bit at a time: within 16 lanes by DPP (rotate by 8, half of
// each row written), across them by the permlane swaps.
__device__ __forceinline__ void swap_bit(uint32_t& a, uint32_t& b, int bit) {
    if (bit == 0) {
        const uint32_t na = (uint32_t)__builtin_amdgcn_update_dpp((int)a, (int)b, 0x128, 0xf, 0xc, false);
        b = (uint32_t)__builtin_amdgcn_update_dpp((int)b, (int)a, 0x128, 0xf, 0x3, false);
        a = na;
    } else if (bit == 1) {
        const auto s = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = s[0];
        b = s[1];
    } else {
        const auto s = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = s[0];
        b = s[1];
    }
}
__device__ __forceinline__ void swap_bit(float& a, float& b, int bit) {
    uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
    swap_bit(x, y, bit);
    a = __uint_as_float(x);
    b = __uint_as_float(y);
}
__device__ __forceinline__ void swap_bit(double& a, double& b, int bit) {
    uint32_t xl = (uint32_t)__double2loint(a), yl = (uint32_t)__double2loint(b);
    uint32_t xh = (uint32_t)__double2hiint(a), yh = (uint32_t)__double2hiint(b);
    swap_bit(xl, yl, bit);
    swap_bit(xh, yh, bit);
    a = __hiloint2double((int)xh, (int)xl);
    b = __hiloint2double((int)yh, (int)yl);
}
template <typename C>
__device__ __forceinline__ void lane_transpose(C (&v)[8]) {
#pragma unroll
    for (int bit = 0; bit < 3; ++bit)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            if (r >> bit & 1) continue;
            swap_bit(v[r].x, v[r | 1 << bit].x, bit);
            swap_bit(v[r].y, v[r | 1 << bit].y, bit);
        }
}

// The y solve of a periodic y for columns in registers: nyp = NCH*L independent
// rows, thread (chunk c, mode m) holding rows c + NCH r, r < L, of its mode.
//   X(ky) = sum_c w_NCH^{c k1} w_nyp^{c k2} [sum_r w_L^{r k2} x(c + NCH r)],  ky = k2 + L k1
// so the length-L transform runs in registers, the real and then the imaginary
// parts are exchanged through LDS (all chunks of one k2 to one thread, S*L
// doubles), and the length-NCH transforms run in registers again; the modes
// are divided by lx + kyy(ky) + lz (1/nyp folded in, the zero mode set to
// zero) and taken back the same way.  A thread takes the IT = L/NCH values
// k2 = c + NCH s.  twy[e] = exp(-2 pi i e/nyp).
template <int NCH, int L, int N>
__device__ __forceinline__ void periodic_ysolve(double2 (&x)[L], double* ex, const double2* twy, const double* kyy,
                                                double lxz, double inv_ny, bool zero_plane, int c, int m, int base,
                                                bool act) {
    constexpr int IT = L / NCH;
    static_assert(L % NCH == 0, "whole second-step items");
    dft_reg<-1, L>(x);
#pragma unroll
    for (int k2 = 1; k2 < L; ++k2) x[k2] = twiddle<-1>(x[k2], twy[c * k2]);
    // slot of (k2, chunk) for this thread's plane and mode
    auto slot = [&](int k2, int cc) { return base + (k2 * NCH + cc) * N + m; };
    auto to_chunks = [&]() {  // x[k2] of chunk c -> x[s*NCH + cc] = chunk cc of k2 = c + NCH s
#pragma unroll
        for (int part = 0; part < 2; ++part) {
            if (act) {
#pragma unroll
                for (int k2 = 0; k2 < L; ++k2) ex[slot(k2, c)] = part ? x[k2].y : x[k2].x;
            }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < IT; ++s)
#pragma unroll
                for (int cc = 0; cc < NCH; ++cc) {
                    const double v = ex[slot(c + NCH * s, cc)];
                    if (part) x[s * NCH + cc].y = v;
                    else x[s * NCH + cc].x = v;
                }
            __syncthreads();
        }
    };
    auto to_rows = [&]() {  // and back
#pragma unroll
        for (int part = 0; part < 2; ++part) {
            if (act) {
#pragma unroll
                for (int s = 0; s < IT; ++s)
#pragma unroll
                    for (int cc = 0; cc < NCH; ++cc)
                        ex[slot(c + NCH * s, cc)] = part ? x[s * NCH + cc].y : x[s * NCH + cc].x;
            }
            __syncthreads();
#pragma unroll
            for (int k2 = 0; k2 < L; ++k2) {
                const double v = ex[slot(k2, c)];
                if (part) x[k2].y = v;
                else x[k2].x = v;
            }
            __syncthreads();
        }
    };
    to_chunks();
#pragma unroll
    for (int s = 0; s < IT; ++s) {
        double2 v[NCH];
#pragma unroll
        for (int cc = 0; cc < NCH; ++cc) v[cc] = x[s * NCH + cc];
        dft_reg<-1, NCH>(v);
#pragma unroll
        for (int k1 = 0; k1 < NCH; ++k1) {
            const int ky = c + NCH * s + L * k1;
            const double f = inv_ny / (lxz + kyy[ky]);
            v[k1] = zero_plane && ky == 0 ? make_double2(0.0, 0.0) : make_double2(v[k1].x * f, v[k1].y * f);
        }
        dft_reg<1, NCH>(v);
#pragma unroll
        for (int cc = 0; cc < NCH; ++cc) x[s * NCH + cc] = v[cc];
    }
    to_rows();
#pragma unroll
    for (int k2 = 1; k2 < L; ++k2) x[k2] = twiddle<1>(x[k2], twy[c * k2]);
    dft_reg<1, L>(x);
}

// What the z kernel reads of a case record, uniform over the workgroup.
template <typename C>
struct ZRec {
    C* spec;
    const double* lu;
    const double* dl;
    const double* du;
    const C* tw2;
    int nym, nzp, R, zero00, nplanes, nch, pp;
};
template <typename C>
__device__ __forceinline__ ZRec<C> zrec_of(const ZPar<C>& z) {
    return ZRec<C>{z.spec, z.lu, z.dl, z.du, z.tw2, z.nym, z.nzp, z.R, z.zero00, z.nplanes, z.nch, z.pp};
}
// the same from a record in memory, held in scalar registers
template <typename T>
__device__ __forceinline__ T* first_lane(T* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return reinterpret_cast<T*>((uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ int first_lane(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <typename C>
__device__ __forceinline__ ZRec<C> zrec_uniform(const ZPar<C>& z) {
    const ZRec<C> r = zrec_of(z);
    return ZRec<C>{first_lane(r.spec), first_lane(r.lu),      first_lane(r.dl),  first_lane(r.du),
                   first_lane(r.tw2),  first_lane(r.nym),     first_lane(r.nzp), first_lane(r.R),
                   first_lane(r.zero00), first_lane(r.nplanes), first_lane(r.nch), first_lane(r.pp)};
}

// Runs the workgroup's items: rec(w, blk) gives the case record of item w and
// its block there, same(w) whether the next item w has the record of the last
// one.  An item's rows load into the registers that the item before frees,
// behind that item's inverse transform and stores.  NCHY: the chunks of a
// periodic y (rows interleaved over them, periodic_ysolve, zy its tables; row
// nym-1, the duplicate of row 0, is neither read nor written: it keeps what the
// forward x kernel left there, and the inverse one takes row 0 in its place),
// or 0 for the wall solve.
template <typename C, int N1, int N2, int BR, int NB, int NCHY, typename Rec, typename Same>
__device__ __forceinline__ void zplane_run(int w0, int total, Rec rec, Same same, const ZyPar<C>* zy,
                                           unsigned char* smem_raw) {
    using Rl = typename CplxT<C>::real;
    constexpr int N = N1 * N2;
    constexpr int L = BR * NB;
    constexpr int SI = BR / N2;  // first-step items per thread and pass
    static_assert(BR % N2 == 0, "items of a thread fill its rows");
    // rows of 16, 32 or 64 modes, eight per second-step item: a wave holds the
    // eight rows of NC whole chunks in both layouts (lane (row, k2), register
    // (chunk, k1); lane (chunk, mode), register row), so the second exchange
    // stays within the wave and out of LDS
    constexpr bool kLane = zplane_lane(N1, N2, BR);
    constexpr int NC = kLane ? 64 / N : 1;
    // LDS position of element (i1, k2) of local row v: with the lane exchange
    // the eight k2 of an i1 take nine slots, which puts the 8 (FP64) lanes of
    // an LDS cycle in distinct banks in both steps and leaves every access of a
    // thread at a constant distance from its first (instruction offsets, no
    // address arithmetic); else the rotated layout, which needs no room
    constexpr int kPad = zplane_pad(N1, N2, BR);
    // and a wave's first-step items are those same rows (BR/N2 = 1 item a thread): both exchanges are the wave's own,
    // in its own slots, and take no workgroup barrier, so the waves run apart and one's arithmetic covers another's
    // LDS and HBM accesses
    auto exchange = [] {
        if constexpr (kLane) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
            __syncthreads();
        }
    };
    auto pos = [](int v, int i1, int k2) { return kLane ? (v * N1 + i1) * kPad + k2 : zsw<N1, N2>(v, i1, k2); };
    C x[NB][BR];
    bool loaded = false;
    for (int w = w0; w < total; w += gridDim.x) {
    int blk;
    const ZRec<C> zp = rec(w, blk);
    const int nym = zp.nym, R = zp.R, nch = NCHY ? NCHY : zp.nch;
    const int nrow = NCHY ? nym - 1 : nym;           // rows transformed
    constexpr int kStep = NCHY ? NCHY * BR : BR;     // rows from one pass to the next
    const int nzs = zp.nzp / 2 + 1;
    const int S1 = N * nch, S = S1 * zp.pp;  // threads per plane, per workgroup
    // opaque, so that no address derived from it is held in a register over the loop
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const bool act = tid < S;
    const int t = min(tid, S - 1);
    C* A = reinterpret_cast<C*>(smem_raw);  // S * BR values: BR rows of every chunk and plane
    double* dls = reinterpret_cast<double*>(A + zplane_slots(N1, N2, BR, S));  // DL(j-1), nch*L
    double* dus = dls + nch * L;                                               // DU(j), nch*L
    C* twl = reinterpret_cast<C*>(dus + nch * L);  // w_n^(i1 k2) at i1*kPad + k2 (lane exchange), or w_n^e, N
    C* twy = twl + N1 * kPad;                      // periodic y: w_nyp^e (and kyy in dls)
    auto twz = [&](int i1, int k2) { return kLane ? twl[i1 * kPad + k2] : twl[i1 * k2]; };
    // HBM accesses are a uniform base and a 32-bit byte offset per thread (one register per address): the
    // workgroup's planes and pivot rows span well under 4 GiB
    const int b0 = blk * zp.pp;
    const long plane = (long)nym * N;

    // this thread's rows of its mode
    const int tp = t / S1;
    const int tr = t - tp * S1;
    const int c = tr / N, m = tr - c * N;
    const int j0 = c * L;
    const int vrow = (tp * nch + c) * BR;
    // second-step items of the lane exchange: rows v0 + 8 cb, cb < NC
    const int v0 = (tid >> 6) * (NC * 8) + ((tid >> 3) & 7), vend = S / N * BR;

    // its transform items: item s covers elements i1 + N1 i2 of local row v, which is row `row` of pass 0, counted over
    // the workgroup's planes (`end`: its plane's last); formed anew at each use (opaque to the
    // compiler) rather than held over the solve
    struct Item {
        int v, i1, row, end;
    };
    auto item = [&](int s) {
        int tt = t;
        asm volatile("" : "+v"(tt));
        const int it = tt + s * S;
        const int v = it / N1;
        const int vc = v / BR;
        int p = 0;
        if (zp.pp > 1) p = vc / nch;
        const int cc = vc - p * nch, q = v - vc * BR;
        return Item{v, it - v * N1, p * nym + (NCHY ? cc + NCHY * q : cc * L + q), p * nym + nrow - 1};
    };
    // rows of pass b of block k (a partial last workgroup loads rows of its last plane again, unstored)
    auto load_rows = [&](int k, int b) {
        const auto base = reinterpret_cast<const Glob<char>*>(gptr(zp.spec) + (long)k * zp.pp * plane);
        const int last = (zp.nplanes - k * zp.pp) * nym - 1;
#pragma unroll
        for (int s = 0; s < SI; ++s) {
            const Item q = item(s);
            const int row = min(min(q.row + b * kStep, q.end), last);
            const uint32_t o = (uint32_t)(row * N + q.i1) * (uint32_t)sizeof(C);
#pragma unroll
            for (int i2 = 0; i2 < N2; ++i2)
                x[b][s * N2 + i2] = gld<C>(reinterpret_cast<const Glob<C>*>(base + o) + N1 * i2);
        }
    };
    double pl[L], plm;
    auto load_pivots = [&](int k) {
        const int kx0 = k * zp.pp / R;
        const auto base = reinterpret_cast<const Glob<char>*>(gptr(zp.lu) + (long)kx0 * nym * nzs);
        int dk = 0, u = k * zp.pp - kx0 * R;
        if (zp.pp > 1) {
            const int pk = min(k * zp.pp + tp, zp.nplanes - 1), kx = pk / R;
            dk = kx - kx0;
            u = pk - kx * R;
        }
        const uint32_t step = (uint32_t)nzs * (uint32_t)sizeof(double);
        uint32_t o = (uint32_t)((dk * nym + j0) * nzs + lu_pos_mu(m, u, R, N)) * (uint32_t)sizeof(double);
        const uint32_t end = o + (uint32_t)(nym - 1 - j0) * step;  // the plane's last row
        auto at = [&](uint32_t e) { return *reinterpret_cast<const Glob<double>*>(base + e); };
        plm = at(j0 > 0 ? o - step : o);
#pragma unroll
        for (int r = 0; r < L; ++r) {
            pl[r] = at(min(o, end));
            o += step;
        }
    };
    if (!kLane || !loaded) __syncthreads();  // the last item has read its tables and rows
    if (!loaded) {
        // tables first: their waits leave the rows' loads in flight
        for (int e = threadIdx.x; e < N; e += blockDim.x) {
            const int i1 = e / N2, k2 = e - i1 * N2;
            twl[kLane ? i1 * kPad + k2 : e] = gld<C>(gptr(zp.tw2) + (kLane ? i1 * k2 : e));
        }
        if constexpr (NCHY != 0) {
            for (int e = threadIdx.x; e < NCHY * L; e += blockDim.x) {
                dls[e] = gptr(zy->kyy)[e];
                twy[e] = gld<C>(gptr(zy->twy2) + e);
            }
        }
        for (int e = threadIdx.x; e < (NCHY ? 0 : nch * L); e += blockDim.x) {
            dls[e] = e > 0 && e < nym ? gptr(zp.dl)[e - 1] : 0.0;
            dus[e] = e < nym - 1 ? gptr(zp.du)[e] : 0.0;
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) load_rows(blk, b);
        __syncthreads();
    }

#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (act) {
#pragma unroll
            for (int s = 0; s < SI; ++s) {
                const Item q = item(s);
                const int v = q.v, i1 = q.i1;
                C w[N2];
#pragma unroll
                for (int i2 = 0; i2 < N2; ++i2) w[i2] = x[b][s * N2 + i2];
                if constexpr (N2 > 1) dft_reg<-1, N2>(w);
                if (!NCHY && q.row + b * BR > q.end) {  // rows past the plane
#pragma unroll
                    for (int i2 = 0; i2 < N2; ++i2) w[i2] = CplxT<C>::make((Rl)0, (Rl)0);
                }
                A[pos(v, i1, 0)] = w[0];
#pragma unroll
                for (int k2 = 1; k2 < N2; ++k2) A[pos(v, i1, k2)] = twiddle<-1>(w[k2], twz(i1, k2));
            }
        }
        if (!NCHY && b == NB - 1) load_pivots(blk);  // in flight over the last second step
        exchange();
        if constexpr (kLane) {
#pragma unroll
            for (int cb = 0; cb < NC; ++cb) {
                const int v = min(v0 + 8 * cb, vend - 1), k2 = tid & 7;
                C w[N1];
#pragma unroll
                for (int i1 = 0; i1 < N1; ++i1) w[i1] = A[pos(v, i1, k2)];
                dft_reg<-1, N1>(w);
#pragma unroll
                for (int k1 = 0; k1 < N1; ++k1) x[b][cb * N1 + k1] = w[k1];
            }
            lane_transpose(x[b]);
        } else {
            if (act) {
                const int items = S * BR / N1;
#pragma unroll 1
                for (int it = t; it < items; it += S) {
                    const int v = it / N2, k2 = it - v * N2;
                    C w[N1];
#pragma unroll
                    for (int i1 = 0; i1 < N1; ++i1) w[i1] = A[pos(v, i1, k2)];
                    dft_reg<-1, N1>(w);
#pragma unroll
                    for (int k1 = 0; k1 < N1; ++k1) A[pos(v, k1, k2)] = w[k1];
                }
            }
            exchange();
#pragma unroll
            for (int q = 0; q < BR; ++q) x[b][q] = A[pos(vrow + q, m / N2, m % N2)];
        }
        exchange();
    }

    if constexpr (NCHY != 0) {
        if constexpr (kLane) __syncthreads();  // every wave's rows have left the slots that the columns exchange through
        const int pk = min(b0 + tp, zp.nplanes - 1), kx = pk / R, kz = R * m + pk - kx * R;
        C f[L];
#pragma unroll
        for (int r = 0; r < L; ++r) f[r] = x[r / BR][r % BR];
        periodic_ysolve<NCHY, L, N>(f, reinterpret_cast<double*>(smem_raw), twy, dls, gptr(zy->kxx)[kx] + gptr(zy->kzz)[kz],
                                    zy->inv_ny, kx == 0 && kz == 0, c, m, tp * NCHY * L * N, act);
#pragma unroll
        for (int r = 0; r < L; ++r) x[r / BR][r % BR] = f[r];
    } else {
    auto solve = [&](auto ends) {
        chunk_ysolve<L, C>([&](int r) -> C& { return x[r / BR][r % BR]; }, pl, plm, dls, dus, nym, j0, c, nch, N, t,
                           act, zp.zero00 && b0 + tp == 0 && m == 0, ends);
    };
    if constexpr (kLane) solve(WaveEnds<64 * kPad * (int)sizeof(C)>{smem_raw});
    else solve(FlatEnds{reinterpret_cast<double2*>(smem_raw), S});
    }

    const int wn = w + gridDim.x;
    loaded = wn < total && same(wn);
    const int kn = blk + gridDim.x;  // an item of the same record

#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if constexpr (kLane) {
            lane_transpose(x[b]);
#pragma unroll
            for (int cb = 0; cb < NC; ++cb) {
                const int v = v0 + 8 * cb, k2 = tid & 7;
                C w[N1];
#pragma unroll
                for (int k1 = 0; k1 < N1; ++k1) w[k1] = x[b][cb * N1 + k1];
                dft_reg<1, N1>(w);
                if (v < vend) {
                    A[pos(v, 0, k2)] = w[0];
#pragma unroll
                    for (int i1 = 1; i1 < N1; ++i1) A[pos(v, i1, k2)] = twiddle<1>(w[i1], twz(i1, k2));
                }
            }
            if (loaded) load_rows(kn, b);
        } else {
            if (act) {
#pragma unroll
                for (int q = 0; q < BR; ++q) A[pos(vrow + q, m / N2, m % N2)] = x[b][q];
            }
            if (loaded) load_rows(kn, b);
            exchange();
            if (act) {
                const int items = S * BR / N1;
#pragma unroll 1
                for (int it = t; it < items; it += S) {
                    const int v = it / N2, k2 = it - v * N2;
                    C w[N1];
#pragma unroll
                    for (int k1 = 0; k1 < N1; ++k1) w[k1] = A[pos(v, k1, k2)];
                    dft_reg<1, N1>(w);
                    A[pos(v, 0, k2)] = w[0];
#pragma unroll
                    for (int i1 = 1; i1 < N1; ++i1) A[pos(v, i1, k2)] = twiddle<1>(w[i1], twz(i1, k2));
                }
            }
        }
        exchange();
        if (act) {
#pragma unroll
            for (int s = 0; s < SI; ++s) {
                const Item q = item(s);
                const int v = q.v, i1 = q.i1;
                C w[N2];
#pragma unroll
                for (int k2 = 0; k2 < N2; ++k2) w[k2] = A[pos(v, i1, k2)];
                if constexpr (N2 > 1) dft_reg<1, N2>(w);
                const int row = q.row + b * kStep;
                if (row <= q.end && row < (zp.nplanes - b0) * nym) {
                    const auto base = reinterpret_cast<Glob<char>*>(gptr(zp.spec) + b0 * plane);
                    const uint32_t o = (uint32_t)(row * N + i1) * (uint32_t)sizeof(C);
                    const auto dst = reinterpret_cast<Glob<C>*>(base + o);
#pragma unroll
                    for (int i2 = 0; i2 < N2; ++i2) gst<C>(dst + N1 * i2, w[i2]);
                }
            }
        }
        if (b + 1 < NB) exchange();
    }
    }
}

template <typename C, int N1, int N2, int BR, int NB>
__global__ void __launch_bounds__(zplane_threads(N1 * N2, NB)) k_zplane(ZPar<C> zp) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    zplane_run<C, N1, N2, BR, NB, 0>(
        xcd_remap(blockIdx.x, gridDim.x), zp.nblocks,
        [&](int w, int& blk) {
            blk = w;
            return zrec_of(zp);
        },
        [](int) { return true; }, nullptr, smem_raw);
}

template <typename C, int N1, int N2, int BR, int NB>
__global__ void __launch_bounds__(zplane_threads(N1 * N2, NB))
kb_zplane(const ZPar<C>* __restrict__ cs, const int* __restrict__ off, const int* __restrict__ idx,
          const int* __restrict__ pnc) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int nc = *pnc;
    int at = -1;  // case of the item in hand
    ZRec<C> r;
    zplane_run<C, N1, N2, BR, NB, 0>(
        xcd_remap(blockIdx.x, gridDim.x), off[nc],
        [&](int w, int& blk) {
            if (at < 0 || w >= off[at + 1]) {
                at = find_case(off, nc, w);
                r = zrec_uniform(cs[idx[at]]);
            }
            blk = w - off[at];
            return r;
        },
        [&](int w) { return w < off[at + 1]; }, nullptr, smem_raw);
}

// periodic y: rows of N1*N2 modes, nyp = NCHY * 8 NB rows.  Up to 512 threads:
// the transforms of 16 values and their twiddles take about 200 registers
// (held to 128, for 1024 threads, they spill 350 bytes a lane).
constexpr int kZpyThreads = 512;
template <int N1, int N2, int NB, int NCHY>
__global__ void __launch_bounds__(kZpyThreads) k_zplane_py(ZyPar<double2> zy) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    zplane_run<double2, N1, N2, 8, NB, NCHY>(
        xcd_remap(blockIdx.x, gridDim.x), zy.z.nblocks,
        [&](int w, int& blk) {
            blk = w;
            return zrec_of(zy.z);
        },
        [](int) { return true; }, &zy, smem_raw);
}

template <typename C, int N1, int N2, int BR>
hipError_t launch_zplane_n(hipStream_t s, int nb, const ZPar<C>& zp, int threads, size_t lds) {
    const dim3 blk(threads);
    auto go = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(resident_grid(k, zp.nblocks, threads, lds)), blk, lds, s, zp);
    };
    if (nb == 1) go(k_zplane<C, N1, N2, BR, 1>);
    else go(k_zplane<C, N1, N2, BR, 2>);
    return hipGetLastError();
}

template <typename C, int N1, int N2, int BR>
hipError_t launch_zplane_batch_n(hipStream_t s, int nb, const ZPar<C>* cs, const int* off, const int* idx,
                                 const int* nc, int grid, int threads, size_t lds) {
    auto go = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(resident_grid(k, grid, threads, lds)), dim3(threads), lds, s, cs, off, idx, nc);
    };
    if (nb == 1) go(kb_zplane<C, N1, N2, BR, 1>);
    else go(kb_zplane<C, N1, N2, BR, 2>);
    return hipGetLastError();
}

// one translation unit per half of the list and precision
#define DFP_ZP_EXTERN(C, a, b, r)                                                                               \
    extern template hipError_t launch_zplane_n<C, a, b, r>(hipStream_t, int, const ZPar<C>&, int, size_t);      \
    extern template hipError_t launch_zplane_batch_n<C, a, b, r>(hipStream_t, int, const ZPar<C>*, const int*,  \
                                                                 const int*, const int*, int, int, size_t);
#define DFP_ZP_INSTANTIATE(C, a, b, r)                                                                          \
    template hipError_t launch_zplane_n<C, a, b, r>(hipStream_t, int, const ZPar<C>&, int, size_t);             \
    template hipError_t launch_zplane_batch_n<C, a, b, r>(hipStream_t, int, const ZPar<C>*, const int*,         \
                                                          const int*, const int*, int, int, size_t);

}  // namespace dfp
