// Block-CSR SpMM: the product of Sparse::KernelMatrixCSR<Kernel_T>::Dot
// (KernelMatrixCSR.hpp:153-227) with the dense block kernels
// (BlockKernels/DenseBlockKernel_Tiny.hpp:160-180, BlockKernels/BlockKernel_Tiny.hpp:
// 156-196).  A pattern of mb x nb blocks (rp, ci) carries one R x C dense block
// per nonzero; for every block row i
//     Y_i <- alpha * sum_{k in row i} A_k X_{ci[k]} + beta * Y_i
// with X_j the C x nrhs chunk at X + j*C*nrhs and Y_i the R x nrhs chunk at
// Y + i*R*nrhs.  Storage orders as the kernel's template flags: A_k row-major
// (a_RM) or column-major; X / Y chunks row-major (x_RM / y_RM: entry (c, h) at
// c*nrhs + h) or transposed (h*C + c).  An empty block row gets Y_i <- beta Y_i
// (WriteYZero, :185-190); alpha == 0 or no nonzeros scales all of Y by beta
// (KernelMatrixCSR.hpp:137-151, 158-162).
//
// GPU layout: a lane group of L lanes (L = R*nrhs rounded up to a power of two,
// at most 64) owns a block row; lane t computes output entries t, t+L, ... of the
// chunk, so lanes of one group read the same A entries (broadcast) and
// neighbouring X entries (coalesced).  The per-lane sum runs over the row's
// blocks in order and over c in order: deterministic.  CSR SpMM bytes per call
// apply with the block sizes: nnzb*(R*C*s + 4) + 4*(mb+1) + nb*C*k*s +
// mb*R*k*s*(1 + [beta != 0]); the gathered X chunks are C*k*s contiguous bytes.
// Memory-bound at every block size the reference instantiates (R, C <= 8:
// 2RCk flops per RCs + Cks bytes stays below 2 flop/byte), so no MFMA.

#include <string>

#include "common.hpp"
#include "krylov.hpp"

namespace tg {

enum BsrBeta : int { kBsrBetaZero = 0, kBsrBetaOne = 1, kBsrBetaGeneric = 2 };

// 1: row-major X / Y chunks use bsr_spmm_vec_kernel (lane = block row x V
// right-hand sides) or bsr_staged_kernel (blocks through LDS); 0: every storage order uses bsr_spmm_kernel (lane = entry).
static int g_bsr_vector = 1;

int bsr_tune_set(const char* key, int32_t value, bool* known) {
    *known = std::string(key) == "bsr_vector";
    if (!*known) return TG_OK;
    if (value != 0 && value != 1) return fail(TG_ERR_INVALID, "tg_tune_set: bsr_vector must be 0 or 1");
    g_bsr_vector = value;
    return TG_OK;
}
int32_t bsr_tune_get(const char* key) { return std::string(key) == "bsr_vector" ? g_bsr_vector : -1; }

template <typename T>
__device__ __forceinline__ T bsr_out(T acc, const T* yp, T alpha, int alpha_one, T beta, int beta_mode) {
    T v = alpha_one ? acc : alpha * acc;
    if (beta_mode == kBsrBetaOne)
        v = v + *yp;
    else if (beta_mode == kBsrBetaGeneric)
        v = v + beta * *yp;
    return v;
}

// CT > 0: C fixed at compile time (loads of a block's C entries issued together).
template <typename T, typename RP, int CT, bool A_RM, bool X_RM, bool Y_RM>
__global__ __launch_bounds__(kBlock) void bsr_spmm_kernel(int mb, int R, int Cr, int k, const RP* __restrict__ rp,
                                                          const int32_t* __restrict__ ci, const T* __restrict__ A,
                                                          T alpha, const T* __restrict__ X, T beta,
                                                          T* __restrict__ Y, int L, int alpha_one, int beta_mode) {
    const int C = CT > 0 ? CT : Cr;
    const int groups = kBlock / L;
    const int t = threadIdx.x % L;
    const int i = blockIdx.x * groups + threadIdx.x / L;
    if (i >= mb) return;
    const RP lo = rp[i], hi = rp[i + 1];
    const int E = R * k;  // entries of the output chunk
    const int64_t RC = (int64_t)R * C, CK = (int64_t)C * k;
    T* __restrict__ Yi = Y + (int64_t)i * E;
    for (int e = t; e < E; e += L) {
        // entry e of the chunk in its storage order -> (r, h)
        const int r = Y_RM ? e / k : e % R;
        const int h = Y_RM ? e % k : e / R;
        T* yp = Yi + e;
        if (hi == lo) {  // WriteYZero: Y_i <- beta Y_i
            *yp = beta_mode == kBsrBetaZero ? T(0) : beta_mode == kBsrBetaOne ? *yp : beta * *yp;
            continue;
        }
        T acc = T(0);
        // two blocks per step (the second clamped to the row's last block and
        // masked), so their index, A and X loads are in flight together
        for (RP kb = lo; kb < hi; kb += 2) {
            const bool two = kb + 1 < hi;
            const RP kb1 = two ? kb + 1 : kb;
            const int64_t j0 = ci[kb], j1 = ci[kb1];
            const T* a0 = A + (int64_t)kb * RC;
            const T* a1 = A + (int64_t)kb1 * RC;
            const T* x0 = X + j0 * CK;
            const T* x1 = X + j1 * CK;
            T s0 = T(0), s1 = T(0);
#pragma unroll
            for (int c = 0; c < (CT > 0 ? CT : 1); ++c) {
                if constexpr (CT > 0) {
                    const int ia = A_RM ? r * C + c : c * R + r;
                    const int ix = X_RM ? c * k + h : h * C + c;
                    s0 += a0[ia] * x0[ix];
                    s1 += a1[ia] * x1[ix];
                }
            }
            if constexpr (CT == 0) {
                for (int c = 0; c < C; ++c) {
                    const int ia = A_RM ? r * C + c : c * R + r;
                    const int ix = X_RM ? c * k + h : h * C + c;
                    s0 += a0[ia] * x0[ix];
                    s1 += a1[ia] * x1[ix];
                }
            }
            acc += s0;
            acc += two ? s1 : T(0);
        }
        *yp = bsr_out(acc, yp, alpha, alpha_one, beta, beta_mode);
    }
}

// Row-major X and Y chunks (the default storage): lane t of a group owns block
// row r and V consecutive right-hand sides h0 .. h0+V-1 (entries t, t+L, ... of
// the R x k/V grid of such tiles), so each block costs it C loads of A and C
// vector loads of V X entries.  k % V == 0 and V-aligned X / Y are checked by the
// host.
template <typename T, typename RP, int CT, int V, bool A_RM>
__global__ __launch_bounds__(kBlock) void bsr_spmm_vec_kernel(int mb, int R, int Cr, int k, const RP* __restrict__ rp,
                                                              const int32_t* __restrict__ ci, const T* __restrict__ A,
                                                              T alpha, const T* __restrict__ X, T beta,
                                                              T* __restrict__ Y, int L, int alpha_one, int beta_mode) {
    const int C = CT > 0 ? CT : Cr;
    const int groups = kBlock / L;
    const int t = threadIdx.x % L;
    const int i = blockIdx.x * groups + threadIdx.x / L;
    if (i >= mb) return;
    const RP lo = rp[i], hi = rp[i + 1];
    const int kv = k / V;
    const int E = R * kv;  // V-wide tiles of the output chunk
    const int64_t RC = (int64_t)R * C, CK = (int64_t)C * k;
    T* __restrict__ Yi = Y + (int64_t)i * R * k;
    for (int e = t; e < E; e += L) {
        const int r = e / kv, h0 = (e % kv) * V;
        T* yp = Yi + (int64_t)r * k + h0;
        T acc[V];
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] = T(0);
        if (hi == lo) {  // WriteYZero: Y_i <- beta Y_i
            T y[V];
            if (beta_mode != kBsrBetaZero) load_vec<T, V>(yp, y);
#pragma unroll
            for (int v = 0; v < V; ++v)
                y[v] = beta_mode == kBsrBetaZero ? T(0) : beta_mode == kBsrBetaOne ? y[v] : beta * y[v];
            store_vec<T, V>(yp, y);
            continue;
        }
        for (RP kb = lo; kb < hi; kb += 2) {
            const bool two = kb + 1 < hi;
            const RP kb1 = two ? kb + 1 : kb;
            const int64_t j0 = ci[kb], j1 = ci[kb1];
            const T* a0 = A + (int64_t)kb * RC;
            const T* a1 = A + (int64_t)kb1 * RC;
            const T* x0 = X + j0 * CK + h0;
            const T* x1 = X + j1 * CK + h0;
            T s0[V], s1[V];
#pragma unroll
            for (int v = 0; v < V; ++v) s0[v] = s1[v] = T(0);
            auto step = [&](int c) {
                const int ia = A_RM ? r * C + c : c * R + r;
                const T av0 = a0[ia], av1 = a1[ia];
                T xv0[V], xv1[V];
                load_vec<T, V>(x0 + (int64_t)c * k, xv0);
                load_vec<T, V>(x1 + (int64_t)c * k, xv1);
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    s0[v] += av0 * xv0[v];
                    s1[v] += av1 * xv1[v];
                }
            };
            if constexpr (CT > 0) {
#pragma unroll
                for (int c = 0; c < CT; ++c) step(c);
            } else {
                for (int c = 0; c < C; ++c) step(c);
            }
#pragma unroll
            for (int v = 0; v < V; ++v) {
                acc[v] += s0[v];
                acc[v] += two ? s1[v] : T(0);
            }
        }
        T y[V];
        if (beta_mode != kBsrBetaZero) load_vec<T, V>(yp, y);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            T out = alpha_one ? acc[v] : alpha * acc[v];
            if (beta_mode == kBsrBetaOne)
                out = out + y[v];
            else if (beta_mode == kBsrBetaGeneric)
                out = out + beta * y[v];
            y[v] = out;
        }
        store_vec<T, V>(yp, y);
    }
}

// Square blocks of side 2, 3, 4, 6 or 8 with row-major chunks.  A group of block rows takes
// its blocks, which lie one after the other in memory, through LDS in chunks of `cap`
// blocks: coalesced loads, each line touched once.  (The kernel above reads a block's rows
// where they lie: lanes 72 bytes apart for 3 x 3 doubles, and by the next block the L1 has
// lost the lines.)  A lane then owns PR rows and V columns of its row's chunk of Y: it loads
// the B x V piece of X once for PR rows, UB blocks in flight, and A comes from LDS, where
// blocks are BS elements apart, an odd number, so that the lanes' rows spread over the
// banks.  Sums in the order of the kernel above.  What bounds it is the chain rp, blocks, X, X
// of a group against the bytes that lie in LDS meanwhile (about 40 MB on the chip at any LDS per
// group), so the X of a lane's first blocks is loaded together with the blocks: 96^3 rows of
// 3 x 3 doubles, k = 4 (637 MB): 191 us before, 193 staged, 158 with that (4.0 TB/s).
// `rows` block rows a workgroup (blockDim.x >= rows * lanes), lanes = (B / PR) * ceil(k / V);
// where V does not divide k the last lane's columns start at k - V and it writes its own.
// A workgroup with far more blocks than planned (kLongChunks chunks) holds a long row, which
// would be one lane group's chain of round trips: it takes its rows one after the other, each
// row's blocks dealt over all lane groups, whose sums meet in LDS (one of 20000 rows with 8000
// blocks of side 4, 5 columns FP32: 1.46 ms in chunks, 0.12 so, 0.73 in the kernel above).
constexpr int kLongChunks = 8;

template <typename T, int B, int V, bool A_RM>
__global__ __launch_bounds__(kBlock) void bsr_staged_kernel(int mb, int k, const void* __restrict__ rp, int rp64,
                                                            const int32_t* __restrict__ ci, const T* __restrict__ A,
                                                            T alpha, const T* __restrict__ X, T beta,
                                                            T* __restrict__ Y, int rows, int lanes, int cap,
                                                            int alpha_one, int beta_mode) {
    constexpr int BB = B * B, BS = BB | 1, PR = B <= 3 ? B : 2, UB = B <= 3 ? 4 : B == 4 ? 2 : 1;
    constexpr int VA = 16 / sizeof(T), LB = 8;  // elements per staging load, loads in flight
    extern __shared__ __align__(16) char lds[];
    T* as = (T*)lds;
    int32_t* cs = (int32_t*)(as + (int64_t)cap * BS);
    const auto at = [&](int i) { return rp64 ? ((const int64_t*)rp)[i] : (int64_t)((const int32_t*)rp)[i]; };
    const int i0 = xcd_swizzle(blockIdx.x, gridDim.x) * rows, i1 = min(i0 + rows, mb);
    const int kv = (k + V - 1) / V;
    const int row = threadIdx.x / lanes, part = threadIdx.x % lanes;
    const int i = i0 + row;
    const bool on = row < rows && i < i1;
    const int r0 = part / kv * PR, hv = part % kv * V, h0 = min(hv, k - V), own = hv - h0;
    const int64_t first = at(i0), end = at(i1);
    const int64_t lo = on ? at(i) : 0, hi = on ? at(i + 1) : 0;
    // Y of the lane's part of row `to`, from its sums
    auto write = [&](int to, bool none, const T (&sum)[PR][V]) {
        T* yp = Y + ((int64_t)to * B + r0) * k + h0;
#pragma unroll
        for (int r = 0; r < PR; ++r) {
            T y[V];
            if (beta_mode != kBsrBetaZero) load_vec_at<T, V>(yp + r * k, y);
#pragma unroll
            for (int v = 0; v < V; ++v) {
                T out = alpha_one ? sum[r][v] : alpha * sum[r][v];
                if (none) out = T(0);  // WriteYZero: Y_i <- beta Y_i
                if (beta_mode == kBsrBetaOne)
                    out = none ? y[v] : out + y[v];
                else if (beta_mode == kBsrBetaGeneric)
                    out = none ? beta * y[v] : out + beta * y[v];
                y[v] = out;
            }
            if (own == 0) {
                store_vec_at<T, V>(yp + r * k, y);
            } else {
#pragma unroll
                for (int v = 1; v < V; ++v)
                    if (v >= own) yp[r * k + v] = y[v];
            }
        }
    };
    if (rows > 1 && end - first > (int64_t)kLongChunks * cap) {
        constexpr int N = PR * V;  // sums of a lane, in as[]: rows * lanes * N (the host's size covers them)
        for (int to = i0; to < i1; ++to) {
            const int64_t from = at(to), till = at(to + 1);
            T sum[PR][V] = {};
            for (int64_t q = from + row; row < rows && q < till; q += rows) {
                const T* xp = X + (int64_t)ci[q] * B * k + h0;
                const T* ap = A + q * BB;
#pragma unroll
                for (int c = 0; c < B; ++c) {
                    T xv[V];
                    load_vec_at<T, V>(xp + c * k, xv);
#pragma unroll
                    for (int r = 0; r < PR; ++r) {
                        const T av = ap[A_RM ? (r0 + r) * B + c : c * B + r0 + r];
#pragma unroll
                        for (int v = 0; v < V; ++v) sum[r][v] += av * xv[v];
                    }
                }
            }
            __syncthreads();
            if (row < rows)
#pragma unroll
                for (int e = 0; e < N; ++e) as[(int)threadIdx.x * N + e] = sum[e / V][e % V];
            __syncthreads();
            if (row == 0) {
                for (int g = 1; g < rows; ++g)
#pragma unroll
                    for (int e = 0; e < N; ++e) sum[e / V][e % V] += as[(g * lanes + part) * N + e];
                write(to, till == from, sum);
            }
        }
        return;
    }
    T acc[PR][V] = {};
    for (int64_t q0 = first; q0 < end; q0 += cap) {
        const int nq = (int)min((int64_t)cap, end - q0), len = nq * BB;
        const T* Aq = A + q0 * BB;
        for (int t = threadIdx.x; t < nq; t += blockDim.x) cs[t] = ci[q0 + t];
        // the lane's blocks in the chunk; the X of its first ones is on its way with the blocks
        const int a = on ? (int)(max(lo, q0) - q0) : 0, b = on ? (int)(min(hi, q0 + nq) - q0) : 0;
        T x[UB][B][V];
        auto fetch = [&](const int32_t (&j)[UB]) {
#pragma unroll
            for (int u = 0; u < UB; ++u) {
                const T* xp = X + (int64_t)j[u] * B * k + h0;
#pragma unroll
                for (int c = 0; c < B; ++c) load_vec_at<T, V>(xp + c * k, x[u][c]);
            }
        };
        int32_t j[UB];
        if (a < b) {
#pragma unroll
            for (int u = 0; u < UB; ++u) j[u] = ci[q0 + min(a + u, b - 1)];
        }
        for (int e0 = threadIdx.x * VA; e0 < len; e0 += LB * VA * blockDim.x) {
            T v[LB][VA];
#pragma unroll
            for (int u = 0; u < LB; ++u)  // the last one overlaps (len >= VA)
                load_vec_at<T, VA>(Aq + min(e0 + u * VA * (int)blockDim.x, len - VA), v[u]);
            if (e0 == (int)threadIdx.x * VA && a < b) fetch(j);
#pragma unroll
            for (int u = 0; u < LB; ++u) {
                const int e = min(e0 + u * VA * (int)blockDim.x, len - VA);
#pragma unroll
                for (int w = 0; w < VA; ++w) as[(e + w) / BB * BS + (e + w) % BB] = v[u][w];
            }
        }
        if ((int)threadIdx.x * VA >= len && a < b) fetch(j);
        __syncthreads();
        for (int kb = a; kb < b; kb += UB) {
            if (kb > a) {
#pragma unroll
                for (int u = 0; u < UB; ++u) j[u] = cs[min(kb + u, b - 1)];
                fetch(j);
            }
#pragma unroll
            for (int u = 0; u < UB; ++u) {
                const T* ap = as + min(kb + u, b - 1) * BS;
                const bool have = kb + u < b;
#pragma unroll
                for (int r = 0; r < PR; ++r) {
                    T sum[V] = {};
#pragma unroll
                    for (int c = 0; c < B; ++c) {
                        const T av = ap[A_RM ? (r0 + r) * B + c : c * B + r0 + r];
#pragma unroll
                        for (int v = 0; v < V; ++v) sum[v] += av * x[u][c][v];
                    }
#pragma unroll
                    for (int v = 0; v < V; ++v) acc[r][v] += have ? sum[v] : T(0);
                }
            }
        }
        __syncthreads();
    }
    if (on) write(i, hi == lo, acc);
}

// Whether blocks go through LDS.  They do where bsr_spmm_vec_kernel has one column a lane (odd k)
// or two (k % 4 == 2), or fewer tiles of four columns than its power of two of lanes, and for
// FP64 blocks of side 4 and 8 from k = 16.  Longer rows (mean over 7) are a longer chain for a
// staged lane, and a small product does not fill the chip to hide it; factors old / staged:
//   rows of 4-7 blocks, 8e4 to 4e5 of them: odd k >= 5 1.0-2.7, k % 4 == 2 FP64 1.0-1.5, FP32
//     1.0-1.7, k = 3 FP64 up to side 6 1.0-1.6 and FP32 up to side 3 1.1-1.4, side 3 FP64 1.0-1.6,
//     side 6 FP64 k >= 8 1.1-1.9, side 8 1.0-2.8.  Not taken: side 2 k = 4 and, FP64, k % 4 == 2
//     (0.9), side 4 FP32 k = 16, 64 (0.6-1.1) and FP64 k = 64 (0.9-1.0), side 6 FP32 k = 8 below 2^18
//     blocks (0.8-1.3), side 8 FP64 k = 6 below 2^17 (0.9).
//   rows of 7-16, k <= 8: 0.5-1.4 at 8e4, 0.6-1.6 at 1.5e5 but for odd k of side 6 and 8 (0.9-1.5)
//     and, from 1.5e5, side 4 and 7 columns of side 3 FP64 (1.1-1.4); at 4e5 1.0-2.5 for odd k, FP32
//     k = 6 from side 3 on, side 3 FP64 but k = 4, k = 3 FP64 of side 6; the same from 2.7e5 on, but
//     FP32 sides 2 and 3 with rows over 11 (0.8-0.9).  k > 16 1.2-2.3 (side 2 FP32, 7e4: 0.8-1.0);
//     k = 9-15 1.0-2.0, but below 2^17 blocks side 3 (0.9-1.0) and even k up to side 6 (0.9-1.2), below 2^18
//     even k of side 3 and FP64 side 6 (0.8-1.0), and rows over 11 of side 2 and 3 (0.5-0.9) and,
//     below 2^17, FP32 of side 4 and 6 (0.7-0.9).
//   below 65536 blocks: k >= 24 1.0-3.1, FP64 side 6 and 8 with odd k and side 6 from k = 12 1.0-1.6;
//     the rest 0.6-1.2 in the kernel (6000 rows of 6, side 6, k = 8 FP32 8.6 against 11.0 us).
//   Side 3 FP64 with 15 of 16 lanes busy (k = 10, 20) 0.8-0.9 for rows of 4-7.
// Rows of 1-3 mean reading past them (0.6-1.2), rows of 27 leave a workgroup few rows (0.5-1.7).
// Other sides (1, 5, 7) keep the mapping above: a staged lane takes one to three whole rows of a
// block, and sides that its rows do not divide were not written.
static bool bsr_staged_pays(int side, int k, bool fp64, int64_t nnzb, int64_t mb) {
    if (k > 64 || nnzb < 32768 || nnzb < 4 * mb || nnzb > 16 * mb) return false;
    const bool longer = nnzb > 7 * mb, longest = nnzb > 11 * mb, many = nnzb >= (1 << 18), some = nnzb >= (1 << 17);
    const bool odd = k % 2 && k >= 5;
    if (nnzb < 65536 && k < 24 && !(fp64 && side >= 6 && (odd || (side == 6 && k >= 12)))) return false;
    const bool enough = nnzb >= (!fp64 && side <= 3 && k < 9 && longest ? 3 << 17 : 1 << 18);
    const int tiles = side * k / (k % 4 == 0 ? 4 : k % 2 == 0 ? 2 : 1);
    int lanes = 1;
    while (lanes < tiles) lanes *= 2;
    if (side == 3 && fp64 && k % 2 == 0 && !longer && 8 * tiles > 7 * lanes) return false;
    if (k % 4) {
        if (k < 3 || (k == 3 && side > (fp64 ? 6 : 3)) || (k % 4 == 2 && side == 2 && fp64)) return false;
        if (!longer) return !(k == 6 && side == 8 && fp64) || some;
        if (enough) return k != 3 ? odd || k > 6 || (fp64 ? side == 3 : side >= 3) : fp64 && side % 3 == 0;
        if (k > 16) return side > 2 || (longest ? fp64 && some : fp64 || some);
        if (k >= 9 && !longest)
            return k % 2 == 0 ? side == 8 || (some && side != 3 && !(side == 6 && fp64)) : side != 3 || some;
        if (k >= 9) return side == 8 || (side == 6 && (fp64 ? odd : some)) || (side == 4 && (fp64 || some));
        if (!odd) return false;
        if (side == 6) return longest ? k == 7 && (fp64 || some) : fp64 || k == 7;
        return side == 8 || (some && (side == 4 ? fp64 || (k == 7 && !longest) : fp64 && side == 3 && k == 7));
    }
    const bool idle = lanes != tiles;
    switch (side) {
        case 3: return fp64 && (!longer || k > 8 || (k == 8 && many));
        case 4: return k >= 16 && (fp64 ? idle || k <= 32 : idle && (!longer || some));
        case 6: return k > 8 ? fp64 || !longest || some || k > 32 : k == 8 && (fp64 ? !longer || many : !longer && many);
        case 8: return k >= 16 && (idle || fp64 || k > 32 || !longer || many);
        default: return false;
    }
}

// The launch of bsr_staged_kernel: 20 KB of LDS a workgroup (12 / 16 / 20 / 24 / 32 / 40 KB,
// the case above: 204 / 172 / 158 / 158 / 160 / 163 us; with 12 or 16 too few lanes of a wave
// have rows), block rows for as many blocks of the mean row (and one more) as that holds, at
// most 256 lanes, in whole waves where there is more than one.
template <typename T, int B>
static int launch_bsr_staged(int mb, int64_t nnzb, int k, const void* rp, int rp64, const int32_t* ci, const T* A,
                             int a_rm, T alpha, const T* X, T beta, T* Y, int alpha_one, int beta_mode, hipStream_t s) {
    constexpr int BS = B * B | 1, PR = B <= 3 ? B : 2, bytes = BS * (int)sizeof(T) + 4;
    int V = (int)(16 / sizeof(T));
    while (V > k) V /= 2;
    const int lanes = B / PR * ((k + V - 1) / V);
    const int64_t mean = (nnzb + mb - 1) / mb + 1;
    int cap = 20 * 1024 / bytes;
    int rows = (int)std::max<int64_t>(1, std::min<int64_t>(kBlock / lanes, cap / mean));
    if (rows * lanes > kWave) rows = std::max(1, rows * lanes / kWave * kWave / lanes);
    cap = (int)std::min<int64_t>(cap, std::max<int64_t>(rows * mean, 8));
    const int threads = (rows * lanes + kWave - 1) / kWave * kWave;
    const dim3 grid((unsigned)((mb + rows - 1) / rows));
    // (a lane's sums of a long row need less: at most 256 lanes of 6 FP64 or 12 FP32 values)
    const size_t shared = std::max((size_t)cap * bytes, (size_t)threads * PR * V * sizeof(T));
#define TG_BSRS(VV)                                                                                             \
    do {                                                                                                        \
        if (a_rm)                                                                                               \
            hipLaunchKernelGGL((bsr_staged_kernel<T, B, VV, true>), grid, dim3(threads), shared, s, mb, k, rp,  \
                               rp64, ci, A, alpha, X, beta, Y, rows, lanes, cap, alpha_one, beta_mode);         \
        else                                                                                                    \
            hipLaunchKernelGGL((bsr_staged_kernel<T, B, VV, false>), grid, dim3(threads), shared, s, mb, k, rp, \
                               rp64, ci, A, alpha, X, beta, Y, rows, lanes, cap, alpha_one, beta_mode);         \
    } while (0)
    if constexpr (sizeof(T) == 4) {
        if (V == 4) {
            TG_BSRS(4);
            TG_LAUNCH_CHECK();
            return TG_OK;
        }
    }
    if (V == 2)
        TG_BSRS(2);
    else
        TG_BSRS(1);
#undef TG_BSRS
    TG_LAUNCH_CHECK();
    return TG_OK;
}

// Y <- beta Y over `count` entries (beta == 0: zero, NaN-free).
template <typename T>
__global__ __launch_bounds__(kBlock) void bsr_scale_kernel(int64_t count, T beta, int beta_mode, T* __restrict__ Y) {
    for (int64_t e = blockIdx.x * (int64_t)kBlock + threadIdx.x; e < count; e += (int64_t)gridDim.x * kBlock)
        Y[e] = beta_mode == kBsrBetaZero ? T(0) : beta * Y[e];
}

// FillLowerTriangleFromUpperTriangle (KernelMatrixCSR.hpp:71-128): for every block
// (i, j) with j < i, the block (j, i) of the upper triangle, transposed.  One
// thread per block row; the upper block is found by binary search in row j from
// its diagonal position (the first column >= j).  Square blocks only.  A lower
// block whose mirror is absent from the pattern is left as it is.
template <typename T, typename RP>
__global__ __launch_bounds__(kBlock) void bsr_fill_lower_kernel(int mb, int R, const RP* __restrict__ rp,
                                                                const int32_t* __restrict__ ci, T* A) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= mb) return;
    const int64_t RR = (int64_t)R * R;
    for (RP kb = rp[i]; kb < rp[i + 1] && ci[kb] < i; ++kb) {
        const int j = ci[kb];
        RP lo = rp[j];
        RP hi = rp[j + 1];
        while (lo < hi && ci[lo] < j) ++lo;  // diagonal position of row j (rows are short)
        // last position in [lo, hi) with column <= i
        RP L = lo, Rr = hi - 1;
        while (L < Rr) {
            const RP M = Rr - (Rr - L) / 2;
            if (ci[M] > i)
                Rr = M - 1;
            else
                L = M;
        }
        if (L >= hi || ci[L] != i) continue;
        const T* from = A + (int64_t)L * RR;
        T* to = A + (int64_t)kb * RR;
        for (int a = 0; a < R; ++a)
            for (int b = 0; b < R; ++b) to[(int64_t)a * R + b] = from[(int64_t)b * R + a];
    }
}

template <typename T, typename RP, int CT>
static void launch_bsr_ct(int a_rm, int x_rm, int y_rm, dim3 grid, hipStream_t s, int mb, int R, int C, int k,
                          const RP* rp, const int32_t* ci, const T* A, T alpha, const T* X, T beta, T* Y, int L,
                          int alpha_one, int beta_mode) {
#define TG_BSR(AR, XR, YR)                                                                                    \
    hipLaunchKernelGGL((bsr_spmm_kernel<T, RP, CT, AR, XR, YR>), grid, dim3(kBlock), 0, s, mb, R, C, k, rp, ci, A, \
                       alpha, X, beta, Y, L, alpha_one, beta_mode)
    const int code = (a_rm ? 4 : 0) | (x_rm ? 2 : 0) | (y_rm ? 1 : 0);
    switch (code) {
        case 0: TG_BSR(false, false, false); break;
        case 1: TG_BSR(false, false, true); break;
        case 2: TG_BSR(false, true, false); break;
        case 3: TG_BSR(false, true, true); break;
        case 4: TG_BSR(true, false, false); break;
        case 5: TG_BSR(true, false, true); break;
        case 6: TG_BSR(true, true, false); break;
        default: TG_BSR(true, true, true); break;
    }
#undef TG_BSR
}

template <typename T, typename RP>
static int bsr_typed(int32_t mb, int64_t nnzb, int32_t R, int32_t C, const RP* rp, const int32_t* ci, const T* A,
                     int a_rm, double alpha_d, const T* X, int x_rm, double beta_d, T* Y, int y_rm, int32_t k,
                     hipStream_t s) {
    const T alpha = (T)alpha_d, beta = (T)beta_d;
    const int beta_mode = beta_d == 0.0 ? kBsrBetaZero : beta_d == 1.0 ? kBsrBetaOne : kBsrBetaGeneric;
    const int64_t total = (int64_t)mb * R * k;
    if (alpha_d == 0.0 || nnzb <= 0) {  // Scale (KernelMatrixCSR.hpp:137-151)
        if (beta_mode == kBsrBetaOne || total == 0) return TG_OK;
        const int grid = (int)std::max<int64_t>(1, std::min<int64_t>((total + kBlock - 1) / kBlock, 8192));
        hipLaunchKernelGGL((bsr_scale_kernel<T>), dim3(grid), dim3(kBlock), 0, s, total, beta, beta_mode, Y);
        TG_LAUNCH_CHECK();
        return TG_OK;
    }
    const int alpha_one = alpha_d == 1.0;
    const bool staged = bsr_staged_pays(R, k, sizeof(T) == 8, nnzb, mb);
    if (x_rm && y_rm && g_bsr_vector && R == C && staged) {
#define TG_BSR_STAGED(BB)                                                                                             \
    case BB:                                                                                                          \
        return launch_bsr_staged<T, BB>(mb, nnzb, k, rp, sizeof(RP) == 8, ci, A, a_rm, alpha, X, beta, Y, alpha_one, \
                                        beta_mode, s)
        switch (R) {
            TG_BSR_STAGED(2);
            TG_BSR_STAGED(3);
            TG_BSR_STAGED(4);
            TG_BSR_STAGED(6);
            TG_BSR_STAGED(8);
        }
#undef TG_BSR_STAGED
    }
    if (x_rm && y_rm && g_bsr_vector) {  // lane = (block row r, V right-hand sides)
        const auto aligned = [&](int bytes) {
            return (uintptr_t)X % bytes == 0 && (uintptr_t)Y % bytes == 0;
        };
        // V * C X values of two blocks stay in registers: V * C <= 16 (FP64) / 32 (FP32)
        const int cap = (int)(128 / sizeof(T));
        int V = 1;
        if (k % 4 == 0 && aligned(4 * (int)sizeof(T)) && 4 * C <= cap)
            V = 4;
        else if (k % 2 == 0 && aligned(2 * (int)sizeof(T)) && 2 * C <= cap)
            V = 2;
        int L = 1;
        while (L < R * (k / V) && L < kWave) L *= 2;
        const int groups = kBlock / L;
        const dim3 grid((unsigned)((mb + groups - 1) / groups));
#define TG_BSRV(CC, VV)                                                                                            \
    do {                                                                                                           \
        if (a_rm)                                                                                                  \
            hipLaunchKernelGGL((bsr_spmm_vec_kernel<T, RP, CC, VV, true>), grid, dim3(kBlock), 0, s, mb, R, C, k, rp, \
                               ci, A, alpha, X, beta, Y, L, alpha_one, beta_mode);                                 \
        else                                                                                                       \
            hipLaunchKernelGGL((bsr_spmm_vec_kernel<T, RP, CC, VV, false>), grid, dim3(kBlock), 0, s, mb, R, C, k,     \
                               rp, ci, A, alpha, X, beta, Y, L, alpha_one, beta_mode);                             \
    } while (0)
#define TG_BSRVC(CC)             \
    case CC:                     \
        if (V == 4)              \
            TG_BSRV(CC, 4);      \
        else if (V == 2)         \
            TG_BSRV(CC, 2);      \
        else                     \
            TG_BSRV(CC, 1);      \
        break;
        switch (C) {
            TG_BSRVC(1)
            TG_BSRVC(2)
            TG_BSRVC(3)
            TG_BSRVC(4)
            TG_BSRVC(6)
            TG_BSRVC(8)
            default:
                if (V == 4)
                    TG_BSRV(0, 4);
                else if (V == 2)
                    TG_BSRV(0, 2);
                else
                    TG_BSRV(0, 1);
        }
#undef TG_BSRVC
#undef TG_BSRV
        TG_LAUNCH_CHECK();
        return TG_OK;
    }
    int L = 1;
    while (L < R * k && L < kWave) L *= 2;
    const int groups = kBlock / L;
    const dim3 grid((unsigned)((mb + groups - 1) / groups));
    switch (C) {
#define TG_BSRC(CC)                                                                                                 \
    case CC:                                                                                                        \
        launch_bsr_ct<T, RP, CC>(a_rm, x_rm, y_rm, grid, s, mb, R, C, k, rp, ci, A, alpha, X, beta, Y, L, alpha_one, \
                                 beta_mode);                                                                        \
        break;
        TG_BSRC(1)
        TG_BSRC(2)
        TG_BSRC(3)
        TG_BSRC(4)
        TG_BSRC(6)
        TG_BSRC(8)
#undef TG_BSRC
        default:
            launch_bsr_ct<T, RP, 0>(a_rm, x_rm, y_rm, grid, s, mb, R, C, k, rp, ci, A, alpha, X, beta, Y, L,
                                    alpha_one, beta_mode);
    }
    TG_LAUNCH_CHECK();
    return TG_OK;
}

}  // namespace tg

using namespace tg;

extern "C" int tg_bsr_spmm(int32_t mb, int32_t nb, int64_t nnzb, int32_t R, int32_t C, const void* rp,
                           tg_dtype rp_type, const int32_t* ci, const void* a, tg_dtype val_type, int32_t a_row_major,
                           double alpha, const void* X, int32_t x_row_major, double beta, void* Y,
                           int32_t y_row_major, int32_t nrhs, void* stream) {
    if (mb < 0 || nb < 0 || nnzb < 0 || R < 1 || C < 1 || nrhs < 0 || R > 64 || C > 64)
        return fail(TG_ERR_INVALID, "tg_bsr_spmm: bad size (block sizes must be in [1, 64])");
    if (val_type != TG_F64 && val_type != TG_F32) return fail(TG_ERR_DTYPE, "tg_bsr_spmm: val_type must be F64/F32");
    if (rp_type != TG_I32 && rp_type != TG_I64) return fail(TG_ERR_DTYPE, "tg_bsr_spmm: rp_type must be I32/I64");
    if (mb == 0 || nrhs == 0) return TG_OK;
    if (!Y) return fail(TG_ERR_INVALID, "tg_bsr_spmm: Y is null");
    const bool compute = alpha != 0.0 && nnzb > 0;
    if (compute) {
        if (!rp || !ci || !a || !X) return fail(TG_ERR_INVALID, "tg_bsr_spmm: rp, ci, values or X is null");
        if (X == Y) return fail(TG_ERR_ALIAS, "tg_bsr_spmm: input and output pointer coincide. Doing nothing.");
    }
    hipStream_t s = as_stream(stream);
    const int ar = a_row_major != 0, xr = x_row_major != 0, yr = y_row_major != 0;
    if (val_type == TG_F64) {
        if (rp_type == TG_I64)
            return bsr_typed<double, int64_t>(mb, nnzb, R, C, (const int64_t*)rp, ci, (const double*)a, ar, alpha,
                                              (const double*)X, xr, beta, (double*)Y, yr, nrhs, s);
        return bsr_typed<double, int32_t>(mb, nnzb, R, C, (const int32_t*)rp, ci, (const double*)a, ar, alpha,
                                          (const double*)X, xr, beta, (double*)Y, yr, nrhs, s);
    }
    if (rp_type == TG_I64)
        return bsr_typed<float, int64_t>(mb, nnzb, R, C, (const int64_t*)rp, ci, (const float*)a, ar, alpha,
                                         (const float*)X, xr, beta, (float*)Y, yr, nrhs, s);
    return bsr_typed<float, int32_t>(mb, nnzb, R, C, (const int32_t*)rp, ci, (const float*)a, ar, alpha,
                                     (const float*)X, xr, beta, (float*)Y, yr, nrhs, s);
}

extern "C" int tg_bsr_fill_lower(int32_t mb, const void* rp, tg_dtype rp_type, const int32_t* ci, int32_t R, void* a,
                                 tg_dtype val_type, void* stream) {
    if (mb < 0 || R < 1 || !rp || !a) return fail(TG_ERR_INVALID, "tg_bsr_fill_lower: bad argument");
    if (val_type != TG_F64 && val_type != TG_F32)
        return fail(TG_ERR_DTYPE, "tg_bsr_fill_lower: val_type must be F64/F32");
    if (rp_type != TG_I32 && rp_type != TG_I64) return fail(TG_ERR_DTYPE, "tg_bsr_fill_lower: rp_type must be I32/I64");
    if (mb == 0) return TG_OK;
    hipStream_t s = as_stream(stream);
    const dim3 grid((unsigned)((mb + kBlock - 1) / kBlock));
#define TG_FL(TT, RR) \
    hipLaunchKernelGGL((bsr_fill_lower_kernel<TT, RR>), grid, dim3(kBlock), 0, s, mb, R, (const RR*)rp, ci, (TT*)a)
    if (val_type == TG_F64) {
        if (rp_type == TG_I64)
            TG_FL(double, int64_t);
        else
            TG_FL(double, int32_t);
    } else {
        if (rp_type == TG_I64)
            TG_FL(float, int64_t);
        else
            TG_FL(float, int32_t);
    }
#undef TG_FL
    TG_LAUNCH_CHECK();
    return TG_OK;
}
