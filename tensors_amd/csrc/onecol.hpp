// Device parts of a one-column Arnoldi step, shared by the single-system GMRES and the
// batched engine: the dots of a tile of rows with the product in front, and the scalars.
#pragma once

#include "common.hpp"

namespace tg {

constexpr int kDdMaxM = 32;            // restart length limit of the one-column step
constexpr int kOneVecs = 4;            // the waves that share a tile's rows
constexpr int kOneRows = 256;          // rows of such a group of waves
constexpr int kOneW = kDdMaxM + 1;     // row length of the staged Hessenberg matrix

// Sums R values per lane over the wave and writes value r to out[at(r)] (at(r) < 0: none).
template <int R, typename At>
__device__ __forceinline__ void wave_sums(double (&v)[R], At at, double* out) {
    const ScatterOut o = wave_scatter_sum<R>(v, 1);
    if (threadIdx.x % o.low == 0)
#pragma unroll
        for (int i = 0; i < ScatterSizes<R>::A; ++i)
            if (i < o.count) {
                const int t = at(o.base + i);
                if (t >= 0) out[t] = v[i];
            }
}

// Place of a lane's register r among the 2j + 2 values [a, b, u.u, u.v], or -1: wave w of
// a group holds a_i (r < NB) and b_i of i = w + 4 (r mod NB), the last one the two others.
template <int NB>
__device__ __forceinline__ int one_place(int r, int j) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) % kOneVecs;
    if (r >= 2 * NB) return w == kOneVecs - 1 ? 2 * j + (r - 2 * NB) : -1;
    const int i = w + kOneVecs * (r < NB ? r : r - NB);
    return i < j ? (r < NB ? i : j + i) : -1;
}

constexpr int kOneNnz = 8;  // nonzeros per thread and chunk of the product
// A row's products of a chunk are added by its thread, in four running sums where there are
// more than kOneShort, and by the thread's wave where there are more than kOneLong: one lane
// would keep the others waiting (100^2 rows, one of them with 2000 nonzeros: 42 ms a solve,
// 9.1 so), and in FP32 a running sum of 2e4 like terms is 1.3e-4 off, the parts 1e-6.
constexpr int kOneShort = 8;
constexpr int kOneLong = 64;

template <typename T, typename RP, int TH, bool SPMV>
struct OneDotsLds {
    T prod[SPMV ? TH * kOneNnz : 1];
    RP srp[SPMV ? TH + 1 : 1];
    T sv[TH], su[TH];
};

// Adds rows [base, base + nr), nr <= TH, to the accumulators of a workgroup of TH threads:
// u = Q_j; v = A u (SPMV; dl / dr: left / right diagonal) written to vslot, or dl z, or
// vslot itself; on a finishing step v = u.  VB vectors are in flight at a time; with VB =
// NB they are loaded before the product.
template <typename T, typename RP, int NB, int VB, int TH, bool SPMV>
__device__ __forceinline__ void one_dots_rows(int base, int nr, int j, int finish, const RP* __restrict__ rp,
                                              const int32_t* __restrict__ ci, const T* __restrict__ a,
                                              const T* __restrict__ dl, const T* __restrict__ dr,
                                              const T* __restrict__ Q, int64_t qstride, const T* __restrict__ z,
                                              T* __restrict__ vslot, OneDotsLds<T, RP, TH, SPMV>& lds,
                                              double (&acc)[2 * NB + 2]) {
    constexpr int EL = kOneNnz, CAP = TH * EL;
    constexpr int RQ = kOneRows / kWave;  // rows per lane
    // wave ids in scalar registers: a basis vector's address is one scalar pair and a lane offset
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int w = wave % kOneVecs, grp = wave / kOneVecs;
    const T* U = Q + (int64_t)j * qstride;
    const int row = base + min((int)threadIdx.x, nr - 1);
    const T uown = U[row];
    T qv[VB][RQ];
    unsigned off[RQ];  // clamped rows
#pragma unroll
    for (int q = 0; q < RQ; ++q) off[q] = (unsigned)min(grp * kOneRows + lane + q * kWave, nr - 1);
    auto load_q = [&](int b0) {  // at clamped vectors
#pragma unroll
        for (int b = 0; b < VB; ++b) {
            const T* qb = Q + (int64_t)max(0, min(w + kOneVecs * (b0 + b), j - 1)) * qstride + base;
#pragma unroll
            for (int q = 0; q < RQ; ++q) qv[b][q] = qb[off[q]];
        }
    };
    if constexpr (VB == NB) load_q(0);  // on their way during the product
    T vown = uown;
    if (SPMV && !finish) {
        for (int i = threadIdx.x; i <= nr; i += TH) lds.srp[i] = rp[base + i];
        __syncthreads();
        const RP l0 = lds.srp[0], l1 = lds.srp[nr];
        T sum = T(0);
        const RP rb = threadIdx.x < nr ? lds.srp[threadIdx.x] : l0, re = threadIdx.x < nr ? lds.srp[threadIdx.x + 1] : l0;
        // (unsigned: cs + CAP may lie past 2^31)
        using UP = typename std::make_unsigned<RP>::type;
        for (UP us = (UP)l0; us < (UP)l1; us += CAP) {
            const RP cs = (RP)us;
            const int cnt = (int)((l1 - cs) < (RP)CAP ? (l1 - cs) : (RP)CAP);
            int32_t c[EL];
            T av[EL], xv[EL];
#pragma unroll
            for (int e = 0; e < EL; ++e) {  // clamped to the chunk's last nonzero
                const RP at = cs + min((int)threadIdx.x + e * TH, cnt - 1);
                c[e] = __builtin_nontemporal_load(ci + at);
                av[e] = a ? __builtin_nontemporal_load(a + at) : T(1);
            }
#pragma unroll
            for (int e = 0; e < EL; ++e) xv[e] = dr ? dr[c[e]] * U[c[e]] : U[c[e]];
#pragma unroll
            for (int e = 0; e < EL; ++e) {
                const int at = threadIdx.x + e * TH;
                if (at < cnt) lds.prod[at] = av[e] * xv[e];
            }
            __syncthreads();
            const int b0 = (int)((rb > cs ? rb : cs) - cs), b1 = (int)((re < cs + cnt ? re : cs + cnt) - cs);
            if (!__any(b1 - b0 > kOneShort)) {  // the plain loop is the shorter one
                for (int l = b0; l < b1; ++l) sum += lds.prod[l];
            } else {
                const bool lng = b1 - b0 > kOneLong;
                if (!lng) sum += lds_sum<T, 1, 1>(lds.prod, b0, b1);
                for (uint64_t left = __ballot(lng); left; left &= left - 1) {  // by the whole wave
                    const int src = __builtin_ctzll(left);
                    const int s0 = __builtin_amdgcn_readlane(b0, src), s1 = __builtin_amdgcn_readlane(b1, src);
                    const T t = group_sum<kWave>(lds_sum<T, kWave, 1>(lds.prod, s0 + lane, s1));
                    if (lane == src) sum += t;
                }
            }
            __syncthreads();
        }
        vown = dl ? dl[row] * sum : sum;
        if (threadIdx.x < nr) vslot[row] = vown;
    } else if (!finish) {
        if (dl) {
            vown = dl[row] * z[row];
            if (threadIdx.x < nr) vslot[row] = vown;
        } else {
            vown = vslot[row];
        }
    }
    lds.su[threadIdx.x] = threadIdx.x < nr ? uown : T(0);
    lds.sv[threadIdx.x] = threadIdx.x < nr ? vown : T(0);
    __syncthreads();
    T uv[RQ], vv[RQ];
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
        uv[q] = lds.su[grp * kOneRows + lane + q * kWave];
        vv[q] = lds.sv[grp * kOneRows + lane + q * kWave];
    }
#pragma unroll
    for (int b0 = 0; b0 < NB; b0 += VB) {
        if constexpr (VB != NB) load_q(b0);
#pragma unroll
        for (int b = 0; b < VB; ++b)
#pragma unroll
            for (int q = 0; q < RQ; ++q) {
                acc[b0 + b] += (double)qv[b][q] * (double)uv[q];
                acc[NB + b0 + b] += (double)qv[b][q] * (double)vv[q];
            }
    }
    if (w == kOneVecs - 1)
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
            acc[2 * NB] += (double)uv[q] * (double)uv[q];
            acc[2 * NB + 1] += (double)uv[q] * (double)vv[q];
        }
    __syncthreads();
}

struct OneScalarLds {
    double sv[2 * kDdMaxM + 2];   // the totals
    double hm[kOneW * kOneW];     // unrotated H, rows 0..j, columns 0..j-1 (j - 1: its first pass)
    double rot[2 * kDdMaxM];      // cs, sn of rotations 0..j-2
    double col[kOneW];            // column j - 1, rotated
    double g[kOneW];              // column j, first pass
    double co, si, carry, kept;   // the new rotation and beta_j, beta_{j-1} after it
    int conv;
};

// The scalars of step j by a workgroup of kBlock threads, from lds.sv, hm and rot: column
// j - 1 completed (hm) and rotated (col) by wave 0, column j's first pass (g, unless
// finishing) by the others.  Synchronised at the end.
__device__ __forceinline__ void one_scalar_core(int j, int finish, const double* __restrict__ beta_jj,
                                                const double* __restrict__ tol, OneScalarLds& lds) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, jj = j - 1;
    // |a|^2 and a.b, by every wave alike
    double aa = 0.0, ab = 0.0;
    const double alane = lane < j ? lds.sv[lane] : 0.0;
    if (lane < j) {
        aa = alane * alane;
        ab = alane * lds.sv[j + lane];
    }
    aa = group_sum<kWave>(aa);
    ab = group_sum<kWave>(ab);
    const double alpha = lds.sv[2 * j], beta = lds.sv[2 * j + 1];
    // |u - Q a|; at a breakdown (u in the span of Q to rounding) at least 2^-52 |u|
    const double rho = j > 0 ? sqrt(fmax(alpha - aa, 0x1p-104 * alpha)) : 1.0;
    const double irho = 1.0 / rho;
    if (j > 0) {
        // column jj completed: its second pass and |u - Q a|
        if (wave == 0 && lane <= j) {
            const double v = lane < j ? lds.hm[lane * kOneW + jj] + alane : rho;
            lds.hm[lane * kOneW + jj] = v;
            lds.col[lane] = v;
        }
        __syncthreads();
    }
    if (wave == 0) {
        if (lane == 0 && j > 0) {
            // Givens on column jj (GMRES.hpp:603-658)
            const double bj = *beta_jj, lim = *tol;
            double xi = lds.col[0];
#pragma unroll 4
            for (int i = 0; i < jj; ++i) {
                const double eta = lds.col[i + 1], co = lds.rot[i], si = lds.rot[kDdMaxM + i];
                lds.col[i] = co * xi + si * eta;
                xi = -si * xi + co * eta;
            }
            const double eta = lds.col[j];
            const double r = sqrt(xi * xi + eta * eta);
            double co, si;
            if (fabs(xi) <= 2.220446049250313e-16 * r) {
                co = 0.0;
                si = 1.0;
            } else {
                const double rinv = 1.0 / r;
                co = fabs(xi) * rinv;
                si = (xi / fabs(xi)) * eta * rinv;
            }
            lds.col[jj] = co * xi + si * eta;
            lds.col[j] = 0.0;
            lds.co = co;
            lds.si = si;
            lds.carry = -si * bj;
            lds.kept = co * bj;
            lds.conv = fabs(-si * bj) <= lim ? 1 : 0;
        }
        if (lane == 0 && j == 0) lds.conv = 0;
    } else if (!finish) {
        // column j, first pass: g_l = (t_l - (H a)_l) / rho, four lanes to a row
        const double tj = j > 0 ? (beta - ab) * irho : beta;
        const int t = threadIdx.x - kWave, part = t % 4;
        for (int l = t / 4; l <= j; l += (kBlock - kWave) / 4) {
            double ha = 0.0;
            for (int i = part; i < j; i += 4) ha += lds.hm[l * kOneW + i] * lds.sv[i];
            ha += shfl_xor(ha, 1);
            ha += shfl_xor(ha, 2);
            if (part == 0) lds.g[l] = ((l < j ? lds.sv[j + l] : tj) - ha) * irho;
        }
    }
    __syncthreads();
}

// Coefficients of q_j and of the next vector from the totals sv, by a workgroup: ca, ce in
// LDS, 1/rho and t_j / rho^2 returned.  Synchronised at the end.
template <typename T>
__device__ __forceinline__ void one_coefs(int j, const double* sv, T* ca, T* ce, T& ir, T& cj) {
    const int lane = threadIdx.x % kWave;
    double aa = 0.0, ab = 0.0;
    if (lane < j) {
        const double ai = sv[lane];
        aa = ai * ai;
        ab = ai * sv[j + lane];
    }
    aa = group_sum<kWave>(aa);
    ab = group_sum<kWave>(ab);
    const double alpha = sv[2 * j], beta = sv[2 * j + 1];
    const double irho = j > 0 ? 1.0 / sqrt(fmax(alpha - aa, 0x1p-104 * alpha)) : 1.0;
    const double tj = j > 0 ? (beta - ab) * irho : beta;
    const double cjd = tj * irho * irho;
    if (threadIdx.x < j) {
        ca[threadIdx.x] = (T)(sv[threadIdx.x] * irho);
        ce[threadIdx.x] = (T)(sv[j + threadIdx.x] * irho - cjd * sv[threadIdx.x]);
    }
    ir = (T)irho;
    cj = (T)cjd;
    __syncthreads();
}

}  // namespace tg
