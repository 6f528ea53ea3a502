// Deterministic column-wise reductions of n x k row-major blocks, shared by
// the solver kernels: thread (c, ro) handles column c of rows ro, ro + rows,
// ...; a fixed LDS tree combines the row lanes of a workgroup into
// partial[block * k + c]; one workgroup then adds the workgroup partials in a
// fixed order.  The result does not depend on scheduling.
#pragma once

#include "common.hpp"

namespace tg {

__device__ __forceinline__ void block_row_range(int n, int& i0, int& i1) {
    const int b = blockIdx.x, B = gridDim.x;
    i0 = (int)((int64_t)n * b / B);
    i1 = (int)((int64_t)n * (b + 1) / B);
}

// Thread layout of the column-blocked elementwise kernels: c = column lane,
// ro = row lane; kBlock / kpad rows are processed per sweep.
struct Lanes {
    int c, ro, rows;
};
__device__ __forceinline__ Lanes lanes_of(int kpad) {
    Lanes L;
    L.c = threadIdx.x % kpad;
    L.ro = threadIdx.x / kpad;
    L.rows = kBlock / kpad;
    return L;
}

// Reduce per-thread partials of the same column over the row lanes (fixed
// tree) and store the workgroup partial partial[block * k + c].
__device__ __forceinline__ void column_partial(double v, const Lanes& L, int k, int kpad, double* partial) {
    __shared__ double sh[kBlock];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int s = L.rows / 2; s > 0; s >>= 1) {
        if (L.ro < s) sh[threadIdx.x] += sh[threadIdx.x + s * kpad];
        __syncthreads();
    }
    if (L.ro == 0 && L.c < k) partial[(int64_t)blockIdx.x * k + L.c] = sh[L.c];
}

// column_partial with the row lanes of a wave combined by cross-lane adds and the waves
// through LDS (two barriers instead of up to nine): for kernels that are short enough for
// the tree's barriers to show.  sh: kBlock doubles of LDS.
__device__ __forceinline__ void column_partial_wave(double v, int k, int kpad, double* sh, double* partial) {
    for (int off = kWave / 2; off >= kpad; off >>= 1) v += shfl_xor(v, off);
    __syncthreads();  // sh may still be read
    sh[threadIdx.x] = v;
    __syncthreads();
    const int step = kpad > kWave ? kpad : kWave;
    if (threadIdx.x < k) {
        double t = sh[threadIdx.x];
        for (int q = step; q < kBlock; q += step) t += sh[q + threadIdx.x];
        partial[(int64_t)blockIdx.x * k + threadIdx.x] = t;
    }
}

// Threads of the one-workgroup kernels that finish a reduction.
constexpr int kFinalThreads = 1024;

// Sum of the B workgroup partials of each column in a fixed order, by one
// workgroup of kFinalThreads threads: thread (c, j), j < J = kFinalThreads / kpad,
// adds partials j, j+J, ... into eight running sums (partial j + qJ + 8mJ goes to
// sum q), combines them in a fixed tree, then a fixed tree over j.  Eight loads
// per thread are in flight at a time, so B = 1024-2048 partials of 32 columns
// take a few memory round trips.
__device__ __forceinline__ double column_total(const double* partial, int B, int k, int kpad, int c, int j,
                                               int J) {
    __shared__ double sh[kFinalThreads];
    double s[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q] = 0.0;
    if (c < k) {
        int b = j;
        for (; b + 7 * J < B; b += 8 * J) {
#pragma unroll
            for (int q = 0; q < 8; ++q) s[q] += partial[(int64_t)(b + q * J) * k + c];
        }
#pragma unroll
        for (int q = 0; q < 7; ++q)  // fewer than 8 left
            if (b + q * J < B) s[q] += partial[(int64_t)(b + q * J) * k + c];
    }
    sh[threadIdx.x] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
    for (int h = J / 2; h > 0; h >>= 1) {
        if (j < h) sh[threadIdx.x] += sh[threadIdx.x + h * kpad];
        __syncthreads();
    }
    const double t = sh[c];
    __syncthreads();
    return t;
}

// Totals of B workgroup partials per column, in a fixed order, by a workgroup of kBlock
// threads that needs them itself: out[0 .. k) in LDS (scratch: kBlock doubles of LDS).
// Thread (c, j) adds partials j, j + J, ... into four or eight running sums, the lanes of a
// wave and then the waves are combined in a fixed tree, so every workgroup that calls it
// gets bitwise the same totals.  Saves the one-workgroup kernel between two passes where
// every workgroup can read the B k values.  What bounds it is the round trips of a thread's
// B / J partials, so more than four of them are read eight at a time, at clamped places (no
// branch between the loads): CG iterations of 10^3 rows and 256 columns, B = 250: 103 us
// with four at a time and branches, 49 so; 12^3 and 192: 105 / 52.  Up to four per thread
// (one to four columns) the conditional loads are the shorter form (96^3 rows, one column,
// an iteration 31.4 against 32.4 us).
__device__ __forceinline__ void block_totals(const double* __restrict__ partial, int B, int k, int kpad, double* out,
                                             double* scratch) {
    const int c = threadIdx.x % kpad, j = threadIdx.x / kpad, J = kBlock / kpad;
    double t = 0.0;
    if (B > 4 * J) {
        constexpr int U = 8;
        double s[U] = {};
        if (c < k)
            for (int b = j; b < B; b += U * J) {
                double w[U];
#pragma unroll
                for (int q = 0; q < U; ++q) w[q] = partial[(int64_t)min(b + q * J, B - 1) * k + c];
#pragma unroll
                for (int q = 0; q < U; ++q)
                    if (b + q * J < B) s[q] += w[q];
            }
        t = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    } else if (c < k) {
        double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (j + q * J < B) s[q] = partial[(int64_t)(j + q * J) * k + c];
        t = (s[0] + s[1]) + (s[2] + s[3]);
    }
    for (int off = kWave / 2; off >= kpad; off >>= 1) t += shfl_xor(t, off);
    scratch[threadIdx.x] = t;
    __syncthreads();
    const int step = kpad > kWave ? kpad : kWave;
    if (threadIdx.x < k) {
        double v = scratch[threadIdx.x];
        for (int q = step; q < kBlock; q += step) v += scratch[q + threadIdx.x];
        out[threadIdx.x] = v;
    }
    __syncthreads();
}

}  // namespace tg
