// Sparse structure work on the GPU: triples -> CSR, transpose, sparse x sparse.
//
// triples -> CSR follows MatrixCSR::FromTriples (MatrixCSR/FromTriples.hpp:3-209):
// entries are bucketed by row, each row is ordered by column (SortInner,
// MatrixCSR/SortInner.hpp:3-49), duplicates (i,j) are merged by summing their
// values when compressQ (PatternCSR/Compress.hpp:81-106), and symmetrizeQ adds
// (j,i,a) for every off-diagonal (i,j,a) (FromTriples.hpp:131-145).  Rows,
// columns and nonzero counts are exactly determined and duplicates are summed in
// input order (deterministic).  Two forms with the same results:
//  * buckets of consecutive rows that a workgroup sorts in LDS (bucket_pays): the
//    triples are dealt to their buckets in one pass, in any order, and every row is
//    ordered by (column, input position), which restores the input's order;
//  * one stable LSD radix sort (rocPRIM) of the keys (row, column) with the triple
//    index as payload, over the bits that occur, for everything else (few long rows,
//    very many triples, buckets that do not fit).
//
// transpose follows MatrixCSR::Op<Trans> (MatrixCSR.hpp:445-490): the
// transposed triples go through the same sort, giving sorted rows.
// sparse x sparse follows MatrixCSR::Dot(MatrixCSR) / PatternCSR::DotBinary_
// (MatrixCSR.hpp:835-921, PatternCSR.hpp:731-839): expand every a_ij * b_jk
// into a triple (i, k), then sort and compress.

#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "common.hpp"
#include "krylov.hpp"

namespace tg {

// Radix keys: row << cb | column, cb = the bits of a column; dropped triples get row m.
__global__ void st_expand_kernel(int64_t count, const int32_t* __restrict__ I, const int32_t* __restrict__ J,
                                 int32_t m, int32_t n, int symmetrize, int cb, uint64_t* __restrict__ keys,
                                 uint32_t* __restrict__ idx, int* __restrict__ bad) {
    const int64_t total = symmetrize ? 2 * count : count;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = e < count ? e : e - count;
        int32_t i = I[t], j = J[t];
        const bool ok = i >= 0 && i < m && j >= 0 && j < n;
        if (!ok) atomicOr(bad, 1);
        uint64_t key = (uint64_t)(uint32_t)m << cb;
        if (ok) {
            if (e < count)
                key = ((uint64_t)(uint32_t)i << cb) | (uint32_t)j;
            else if (i != j)  // transposed copy; the diagonal is not duplicated
                key = ((uint64_t)(uint32_t)j << cb) | (uint32_t)i;
        }
        keys[e] = key;
        idx[e] = (uint32_t)e;
    }
}

// head[e] = 1 where a new output entry starts (every entry when not compressing);
// dropped triples (row m) sort last and are never heads.
__global__ void st_heads_kernel(int64_t total, const uint64_t* __restrict__ keys, int compress, uint64_t end,
                                int64_t* __restrict__ head) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t k = keys[e];
        int64_t h = 0;
        if (k < end) h = (!compress || e == 0 || keys[e - 1] != k) ? 1 : 0;
        head[e] = h;
    }
}

// Writes column indices and (summed) values; counts entries per row.
template <typename T>
__global__ void st_write_kernel(int64_t total, const uint64_t* __restrict__ keys, const uint32_t* __restrict__ idx,
                                const int64_t* __restrict__ head, const int64_t* __restrict__ pos, int64_t count,
                                int cb, const T* __restrict__ V, int compress, int32_t* __restrict__ ci, T* __restrict__ val,
                                int64_t* __restrict__ rowcnt) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        if (!head[e]) continue;
        const uint64_t k = keys[e];
        const int64_t p = pos[e];
        ci[p] = (int32_t)(k & ((1ull << cb) - 1));
        atomicAdd((unsigned long long*)&rowcnt[k >> cb], 1ull);
        if (V) {
            const uint32_t t0 = idx[e];
            T s = V[t0 < count ? t0 : t0 - count];
            if (compress)
                for (int64_t f = e + 1; f < total && keys[f] == k; ++f) {
                    const uint32_t t = idx[f];
                    s += V[t < count ? t : t - count];
                }
            val[p] = s;
        }
    }
}

template <typename RP>
__global__ void st_rp_kernel(int32_t m, const int64_t* __restrict__ scanned, RP* __restrict__ rp,
                             int64_t* __restrict__ nnz) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i <= m; i += (int64_t)gridDim.x * blockDim.x) {
        rp[i] = (RP)scanned[i];
        if (i == m) *nnz = scanned[i];
    }
}

__global__ void st_zero64_kernel(int64_t count, int64_t* __restrict__ a, int* __restrict__ flag = nullptr) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        a[i] = 0;
    if (flag && blockIdx.x == 0 && threadIdx.x == 0) *flag = 0;
}

// Bits that hold 0 .. count - 1 (at least one).
static int bits_of(int64_t count) {
    int b = 1;
    while (b < 32 && ((int64_t)1 << b) < count) ++b;
    return b;
}

static int grid_of(int64_t count) {
    return (int)std::max<int64_t>(1, std::min<int64_t>((count + 255) / 256, 16384));
}

// Workspace layout of from_triples.
struct TriplesWs {
    uint64_t* keys[2];
    uint32_t* idx[2];
    int64_t* head;
    int64_t* pos;
    int64_t* rowcnt;  // m + 1
    int64_t* rowscan; // m + 1
    int64_t* nnz;
    int* bad;
    void* temp;
    size_t temp_bytes;
    size_t total_bytes;
};

static size_t triples_ws(int64_t count, int32_t m, int symmetrize, char* base, TriplesWs* out) {
    const int64_t total = symmetrize ? 2 * count : count;
    size_t sort_tmp = 0, scan_tmp = 0, scan_tmp2 = 0;
    (void)rocprim::radix_sort_pairs(nullptr, sort_tmp, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint32_t*)nullptr,
                              (uint32_t*)nullptr, (size_t)std::max<int64_t>(total, 1), 0, 64);
    (void)rocprim::exclusive_scan(nullptr, scan_tmp, (const int64_t*)nullptr, (int64_t*)nullptr, (int64_t)0,
                            (size_t)std::max<int64_t>(total, 1), rocprim::plus<int64_t>());
    (void)rocprim::exclusive_scan(nullptr, scan_tmp2, (const int64_t*)nullptr, (int64_t*)nullptr, (int64_t)0,
                            (size_t)m + 1, rocprim::plus<int64_t>());
    const size_t tmp = std::max(sort_tmp, std::max(scan_tmp, scan_tmp2));
    size_t off = 0;
    auto take = [&](size_t b) {
        const size_t o = off;
        off += align256(std::max<size_t>(b, 8));
        return base ? (void*)(base + o) : nullptr;
    };
    TriplesWs w;
    w.keys[0] = (uint64_t*)take(8 * (size_t)total);
    w.keys[1] = (uint64_t*)take(8 * (size_t)total);
    w.idx[0] = (uint32_t*)take(4 * (size_t)total);
    w.idx[1] = (uint32_t*)take(4 * (size_t)total);
    w.head = (int64_t*)take(8 * (size_t)total);
    w.pos = (int64_t*)take(8 * (size_t)total);
    w.rowcnt = (int64_t*)take(8 * ((size_t)m + 1));
    w.rowscan = (int64_t*)take(8 * ((size_t)m + 1));
    w.nnz = (int64_t*)take(8);
    w.bad = (int*)take(8);
    w.temp = take(tmp);
    w.temp_bytes = tmp;
    w.total_bytes = off;
    if (out) *out = w;
    return off;
}

// The number of entries and the two flags, neighbours in the workspace, in one copy;
// synchronises s.
static int triples_found(const TriplesWs& w, int64_t* nnz, int* bad, int* unfit, hipStream_t s) {
    const size_t span = (size_t)((char*)(w.bad + 2) - (char*)w.nnz);
    char found[512];
    if (span > sizeof(found)) return fail(TG_ERR_INVALID, "internal: workspace layout");
    TG_HIP(hipMemcpyAsync(found, w.nnz, span, hipMemcpyDeviceToHost, s));
    TG_HIP(hipStreamSynchronize(s));
    std::memcpy(nnz, found, 8);
    std::memcpy(bad, found + span - 8, 4);
    std::memcpy(unfit, found + span - 4, 4);
    return TG_OK;
}

// ---------------------------------------------------------------------------
// Bucket form.  The 64-bit radix sort moved 12 bytes a triple through memory eight times
// (10.5 M triples of a 96^3 grid's edges: eight passes of 99 us, 1353 us in all).  Here a
// triple moves twice: to its bucket of rows, and, sorted and merged in LDS, out:
//   bk_hist     triples per bucket
//   bk_offsets  exclusive scan of them (one workgroup)
//   bk_deal     every workgroup deals a tile of triples to the buckets: ranks from LDS
//               counters, one global reservation per tile and bucket
//   bk_sort     a workgroup per bucket: rows by an LDS count, a row's triples by their rank
//               in (column, input position), duplicates summed in that order; merged
//               entries to the bucket's place of a temporary, row starts within the bucket
//   bk_offsets  scan of the merged counts
//   bk_out      copies each bucket's entries to the result and writes its row pointers
// The same case takes 348 us (580 shuffled, the deal 239 of it for 74).  A bucket that does not fit (more than
// kBkCap triples, or a row of more than kBkRow) raises a flag, and the radix form runs
// instead: too many triples before any is dealt, with the kernels that follow returning at
// once.  Radix form alone (64 bits) / with the attempt in front: 1.05e7 triples with a row of
// 1e4 1851 / 1646 us, 2e6 602 / 558, 3e5 343 / 390; rows of up to kBkRow stay in the buckets
// (3e5 triples, one row of 700: 246 / 121 us, of 1400 254 / 165).
// ---------------------------------------------------------------------------
constexpr int kBkThreads = 1024;
constexpr int kBkCap = 3072;        // triples of a bucket (75 KB of LDS: two workgroups a CU)
constexpr int kBkRowBits = 11;
constexpr int kBkRows = 1 << kBkRowBits;  // rows of a bucket
constexpr int kBkIdxBits = 24;      // input positions
constexpr int kBkColBits = 64 - kBkRowBits - kBkIdxBits;
constexpr int kBkRow = 1536;        // triples of a row (ranked against each other)
constexpr int kBkMeanRow = 128;     // ... on average
constexpr int kBkMost = 8192;       // buckets
constexpr int kBkTarget = 1536;     // triples of a bucket on average (up to 2048 where kBkMost binds)
constexpr int kBkPer = 8;           // triples per thread of a tile
constexpr int kBkTile = kBkThreads * kBkPer;

struct BucketPlan {
    int buckets = 0, rows = 0;  // 0 buckets: the radix form
};

// Whether the triples go through buckets: the average row is short (rows of more than kBkRow
// would not fit), a bucket holds a good workgroup's work, and there are not too many.
// Few triples stay with the radix form, whose passes are then launches only.
// A triple travels as one word: row in its bucket, column, input position.
static BucketPlan bucket_plan(int64_t total, int32_t m, int32_t cols) {
    BucketPlan P;
    if (total < 4096 || m < 1 || total / m > kBkMeanRow || total > ((int64_t)1 << kBkIdxBits) ||
        cols > ((int64_t)1 << kBkColBits))
        return P;
    // two a CU if few (small buckets hold denser ranges of rows: 64 triples on average up to 48
    // times that)
    const int64_t target = std::min<int64_t>(kBkTarget, std::max<int64_t>(64, total / 512));
    int64_t nb = std::max((total + target - 1) / target, ((int64_t)m + kBkRows - 1) / kBkRows);
    if (nb > kBkMost && total <= (int64_t)kBkMost * 2048 && m <= (int64_t)kBkMost * kBkRows) nb = kBkMost;
    if (nb > kBkMost || nb * 4 > total) return P;  // the bucket arrays live in 8 bytes a triple
    P.rows = (int)(((int64_t)m + nb - 1) / nb);
    P.buckets = (int)(((int64_t)m + P.rows - 1) / P.rows);
    return P;
}

// Triple e (e >= count: the transposed copy): false if dropped or out of range.
__device__ __forceinline__ bool bk_triple(int64_t e, int64_t count, const int32_t* __restrict__ I,
                                          const int32_t* __restrict__ J, int32_t m, int32_t n, int32_t& r, int32_t& c,
                                          bool& bad) {
    const bool copy = e >= count;
    const int32_t i = I[copy ? e - count : e], j = J[copy ? e - count : e];
    if (i < 0 || i >= m || j < 0 || j >= n) {
        bad = true;
        return false;
    }
    r = copy ? j : i;
    c = copy ? i : j;
    return !(copy && i == j) && r < m;
}

// Adds the lanes with `on` to the LDS counters h[b]; returns each lane's rank there.  Two
// rounds take the lanes that share the first lane's counter together (triples that come in
// mesh order hit one or two counters per wave, 64 times each), the rest go one by one.
// All lanes of the wave call it.
__device__ __forceinline__ uint32_t bk_count(uint32_t* h, int b, bool on) {
    const int lane = threadIdx.x % kWave;
    uint32_t rank = 0;
#pragma unroll
    for (int round = 0; round < 2; ++round) {
        const uint64_t left = __ballot(on);
        if (!left) return rank;
        const int b0 = __builtin_amdgcn_readlane(b, __builtin_ctzll(left));
        const uint64_t same = __ballot(on && b == b0);
        if (on && b == b0) {
            uint32_t base = 0;
            const int first = __builtin_ctzll(same);
            if (lane == first) base = atomicAdd(&h[b0], (uint32_t)__popcll(same));
            base = __builtin_amdgcn_readlane(base, first);
            rank = base + (uint32_t)__popcll(same & ((1ull << lane) - 1));
            on = false;
        }
    }
    if (on) rank = atomicAdd(&h[b], 1u);
    return rank;
}

__global__ void bk_clear_kernel(int nb, uint32_t* __restrict__ hist, int* __restrict__ flags) {
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < nb; b += gridDim.x * blockDim.x) hist[b] = 0;
    if (blockIdx.x == 0 && threadIdx.x < 2) flags[threadIdx.x] = 0;
}

__global__ __launch_bounds__(kBkThreads) void bk_hist_kernel(int64_t count, int64_t total, const int32_t* __restrict__ I,
                                                             const int32_t* __restrict__ J, int32_t m, int32_t n,
                                                             int rows, int buckets, uint32_t* __restrict__ hist,
                                                             int* __restrict__ bad) {
    __shared__ uint32_t h[kBkMost];
    for (int b = threadIdx.x; b < buckets; b += kBkThreads) h[b] = 0;
    __syncthreads();
    bool wrong = false;
    for (int64_t e0 = blockIdx.x * (int64_t)kBkThreads; e0 < total; e0 += (int64_t)gridDim.x * kBkThreads) {
        const int64_t e = e0 + threadIdx.x;
        int32_t r = 0, c;
        const bool on = e < total && bk_triple(e, count, I, J, m, n, r, c, wrong);
        (void)bk_count(h, r / rows, on);
    }
    if (wrong) atomicOr(bad, 1);
    __syncthreads();
    for (int b = threadIdx.x; b < buckets; b += kBkThreads)
        if (h[b]) atomicAdd(&hist[b], h[b]);
}

// Flags of a run that does not fit, in one word: a bucket of more than kBkCap triples, known
// before any triple is dealt (the kernels after it then return at once), or a row of more
// than kBkRow, found while sorting.
constexpr int kBkCrowded = 1, kBkLongRow = 2;

// off[0 .. nb] = exclusive scan of cnt[0 .. nb), nb <= kBkMost; cursor (if given) = off;
// unfit (if given): kBkCrowded where a count is more than kBkCap.
__global__ __launch_bounds__(kBkThreads) void bk_offsets_kernel(int nb, const uint32_t* __restrict__ cnt,
                                                                uint32_t* __restrict__ off,
                                                                uint32_t* __restrict__ cursor,
                                                                int64_t* __restrict__ sum, int* __restrict__ unfit) {
    constexpr int PER = kBkMost / kBkThreads;
    __shared__ uint32_t wsum[kBkThreads / kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    uint32_t v[PER], tot = 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int b = threadIdx.x * PER + q;
        v[q] = b < nb ? cnt[b] : 0;
        tot += v[q];
        if (unfit && v[q] > (uint32_t)kBkCap) atomicOr(unfit, kBkCrowded);
    }
    uint32_t inc = tot;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, kWave);
        if (lane >= o) inc += t;
    }
    if (lane == kWave - 1) wsum[wave] = inc;
    __syncthreads();
    uint32_t run = inc - tot;
    for (int w = 0; w < wave; ++w) run += wsum[w];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int b = threadIdx.x * PER + q;
        if (b < nb) {
            off[b] = run;
            if (cursor) cursor[b] = run;
        }
        run += v[q];
        if (b == nb - 1) {
            off[nb] = run;
            if (sum) *sum = run;
        }
    }
}

// A triple's word: row in its bucket | column | input position.
__device__ __forceinline__ uint64_t bk_word(int row, int32_t col, int64_t e) {
    return ((uint64_t)(uint32_t)row << (kBkColBits + kBkIdxBits)) | ((uint64_t)(uint32_t)col << kBkIdxBits) | (uint64_t)e;
}
__device__ __forceinline__ int bk_row(uint64_t w) { return (int)(w >> (kBkColBits + kBkIdxBits)); }
__device__ __forceinline__ int32_t bk_col(uint64_t w) {
    return (int32_t)((w >> kBkIdxBits) & (((uint64_t)1 << kBkColBits) - 1));
}

template <typename T>
struct alignas(16) BkItem {  // one 16-byte store: shuffled triples are bound by the number of them
    uint64_t word;
    T val;
};

// out: BkItem<T> with values, plain words without.
template <typename T>
__global__ __launch_bounds__(kBkThreads) void bk_deal_kernel(int64_t count, int64_t total, const int32_t* __restrict__ I,
                                                             const int32_t* __restrict__ J, const T* __restrict__ V,
                                                             int32_t m, int32_t n, int rows, int buckets,
                                                             uint32_t* __restrict__ cursor, void* __restrict__ out,
                                                             const int* __restrict__ unfit) {
    const int stop = *unfit;  // (its load is not waited for here)
    __shared__ uint32_t h[kBkMost];
    for (int b = threadIdx.x; b < buckets; b += kBkThreads) h[b] = 0;
    __syncthreads();
    int32_t r[kBkPer], c[kBkPer];
    uint32_t rank[kBkPer];
    const int64_t e0 = blockIdx.x * (int64_t)kBkTile + threadIdx.x;
    bool bad = false;
#pragma unroll
    for (int q = 0; q < kBkPer; ++q) {
        const int64_t e = e0 + q * kBkThreads;
        int32_t rr = 0, cc = 0;
        const bool on = e < total && bk_triple(e, count, I, J, m, n, rr, cc, bad);
        rank[q] = bk_count(h, rr / rows, on);
        r[q] = on ? rr : -1;
        c[q] = cc;
    }
    if (stop) return;
    __syncthreads();
    for (int b = threadIdx.x; b < buckets; b += kBkThreads)
        if (h[b]) h[b] = atomicAdd(&cursor[b], h[b]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kBkPer; ++q) {
        if (r[q] < 0) continue;
        const int64_t e = e0 + q * kBkThreads;
        const int b = r[q] / rows;
        const uint32_t at = h[b] + rank[q];
        const uint64_t word = bk_word(r[q] - b * rows, c[q], e);
        if (V)
            ((BkItem<T>*)out)[at] = BkItem<T>{word, V[e < count ? e : e - count]};
        else
            ((uint64_t*)out)[at] = word;
    }
}

// Exclusive scan of v[0 .. n) in LDS (n <= 4 kBkThreads), v[n] = the total.
__device__ __forceinline__ void bk_scan(uint32_t* v, int n) {
    __shared__ uint32_t wsum[kBkThreads / kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, b0 = 4 * threadIdx.x;
    uint32_t x[4], tot = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        x[q] = b0 + q < n ? v[b0 + q] : 0;
        tot += x[q];
    }
    uint32_t inc = tot;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, kWave);
        if (lane >= o) inc += t;
    }
    if (lane == kWave - 1) wsum[wave] = inc;
    __syncthreads();
    uint32_t run = inc - tot;
    for (int w = 0; w < wave; ++w) run += wsum[w];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (b0 + q < n) v[b0 + q] = run;
        run += x[q];
    }
    if (threadIdx.x == kBkThreads - 1) v[n] = run;  // the last thread's run covers all
    __syncthreads();
}

template <typename T>
__global__ __launch_bounds__(kBkThreads, 8) void bk_sort_kernel(int32_t m, int rows, const uint32_t* __restrict__ off,
                                                                const void* __restrict__ in, int has_val, int compress,
                                                                int32_t* __restrict__ tci, T* __restrict__ tval,
                                                                uint32_t* __restrict__ rowoff,
                                                                uint32_t* __restrict__ merged,
                                                                int* __restrict__ unfit) {
    constexpr int PER = kBkCap / kBkThreads;
    __shared__ uint64_t key[kBkCap], sorted[kBkCap];  // words by row, then sorted
    __shared__ uint16_t first[kBkCap];                // 1 where an entry starts
    __shared__ uint32_t start[kBkRows + 1], head[kBkCap + 1];
    __shared__ int toolong;
    const int stop = *unfit & kBkCrowded;  // set in an earlier launch: the same for all
    T* vals = (T*)key;  // the words by row are done with when the values are placed
    const int b = blockIdx.x, r0 = b * rows, nr = min(rows, m - r0);
    const uint32_t base = off[b];
    const int cnt = (int)(off[b + 1] - base);
    if (stop) return;
    for (int i = threadIdx.x; i < nr; i += kBkThreads) start[i] = 0;
    if (threadIdx.x == 0) toolong = 0;
    __syncthreads();
    uint64_t k[PER];
    T v[PER];
    int r[PER];
    uint32_t at[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int i = threadIdx.x + q * kBkThreads;
        r[q] = -1;
        v[q] = T(0);
        if (i < cnt) {
            if (has_val) {
                const BkItem<T> x = ((const BkItem<T>*)in)[base + i];
                k[q] = x.word;
                v[q] = x.val;
            } else {
                k[q] = ((const uint64_t*)in)[base + i];
            }
            r[q] = bk_row(k[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < PER; ++q)
        if (r[q] >= 0) at[q] = atomicAdd(&start[r[q]], 1u);
    __syncthreads();
    for (int i = threadIdx.x; i < nr; i += kBkThreads)
        if (start[i] > kBkRow) toolong = 1;
    __syncthreads();
    if (toolong) {  // block-uniform
        if (threadIdx.x == 0) {
            atomicOr(unfit, kBkLongRow);
            merged[b] = 0;
        }
        return;
    }
    bk_scan(start, nr);
#pragma unroll
    for (int q = 0; q < PER; ++q)
        if (r[q] >= 0) key[at[q] + start[r[q]]] = k[q];
    __syncthreads();
    // a triple's rank in its row: the words differ, so the ranks do
#pragma unroll
    for (int q = 0; q < PER; ++q)
        if (r[q] >= 0) {
            const int s0 = start[r[q]], s1 = start[r[q] + 1];
            uint32_t rank = 0;
#pragma unroll 4
            for (int t = s0; t < s1; ++t) rank += key[t] < k[q] ? 1 : 0;
            at[q] = s0 + rank;
            sorted[at[q]] = k[q];
        }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q)
        if (r[q] >= 0) vals[at[q]] = v[q];
    // an entry starts where row or column changes
    for (int t = threadIdx.x; t < cnt; t += kBkThreads) {
        const int f = !compress || t == 0 || (sorted[t] >> kBkIdxBits) != (sorted[t - 1] >> kBkIdxBits) ? 1 : 0;
        head[t] = f;
        first[t] = (uint16_t)f;
    }
    __syncthreads();
    bk_scan(head, cnt);
    for (int t = threadIdx.x; t < cnt; t += kBkThreads)
        if (first[t]) {
            const uint32_t o = base + head[t];
            tci[o] = bk_col(sorted[t]);
            if (has_val) {
                T sum = vals[t];
                for (int u = t + 1; u < cnt && !first[u]; ++u) sum += vals[u];
                tval[o] = sum;
            }
        }
    for (int i = threadIdx.x; i < nr; i += kBkThreads) rowoff[r0 + i] = head[start[i]];
    if (threadIdx.x == 0) merged[b] = head[cnt];
}

template <typename T, typename RP>
__global__ __launch_bounds__(256) void bk_out_kernel(int32_t m, int rows, const uint32_t* __restrict__ off,
                                                     const uint32_t* __restrict__ moff,
                                                     const uint32_t* __restrict__ rowoff,
                                                     const int32_t* __restrict__ tci, const T* __restrict__ tval,
                                                     RP* __restrict__ rp, int32_t* __restrict__ ci, T* __restrict__ val,
                                                     const int* __restrict__ unfit) {
    const int stop = *unfit;
    const int b = blockIdx.x, r0 = b * rows, nr = min(rows, m - r0);
    const uint32_t src = off[b], dst = moff[b];
    const int cnt = (int)(moff[b + 1] - dst);
    if (stop) return;
    for (int i = threadIdx.x; i < nr; i += 256) rp[r0 + i] = (RP)(dst + rowoff[r0 + i]);
    if (b == (int)gridDim.x - 1 && threadIdx.x == 0) rp[m] = (RP)(dst + cnt);
    for (int t = threadIdx.x; t < cnt; t += 256) {
        ci[dst + t] = tci[src + t];
        if (tval) val[dst + t] = tval[src + t];
    }
}

// The bucket form; *unfit != 0 when a bucket did not fit (nothing was written).
template <typename T>
static int bucket_triples(const BucketPlan& P, int64_t count, int64_t total, const int32_t* I, const int32_t* J,
                          const T* V, int32_t m, int32_t n, int compress, void* rp_out, tg_dtype rp_type,
                          int32_t* ci_out, T* val_out, const TriplesWs& w, int64_t* nnz, int* bad, int* unfit,
                          hipStream_t s) {
    const int nb = P.buckets;
    uint32_t* hist = (uint32_t*)w.pos;      // then the cursors, then the merged counts
    uint32_t* off = hist + nb;              // nb + 1
    uint32_t* moff = off + nb + 1;          // nb + 1
    void* items = w.keys[0];                // 16 bytes a triple: both key arrays, one after the other
    int32_t* tci = (int32_t*)w.idx[1];
    T* tval = V ? (T*)w.head : nullptr;
    uint32_t* rowoff = (uint32_t*)w.rowcnt;
    hipLaunchKernelGGL(bk_clear_kernel, dim3(grid_of(nb)), dim3(256), 0, s, nb, hist, w.bad);
    const int hgrid = (int)std::max<int64_t>(1, std::min<int64_t>(512, (total + kBkTile - 1) / kBkTile));
    hipLaunchKernelGGL(bk_hist_kernel, dim3(hgrid), dim3(kBkThreads), 0, s, count, total, I, J, m, n, P.rows, nb, hist,
                       w.bad);
    hipLaunchKernelGGL(bk_offsets_kernel, dim3(1), dim3(kBkThreads), 0, s, nb, (const uint32_t*)hist, off, hist,
                       (int64_t*)nullptr, w.bad + 1);
    hipLaunchKernelGGL((bk_deal_kernel<T>), dim3((unsigned)((total + kBkTile - 1) / kBkTile)), dim3(kBkThreads), 0, s,
                       count, total, I, J, V, m, n, P.rows, nb, hist, items, (const int*)(w.bad + 1));
    hipLaunchKernelGGL((bk_sort_kernel<T>), dim3(nb), dim3(kBkThreads), 0, s, m, P.rows, (const uint32_t*)off,
                       (const void*)items, V ? 1 : 0, compress, tci, tval, rowoff, hist, w.bad + 1);
    hipLaunchKernelGGL(bk_offsets_kernel, dim3(1), dim3(kBkThreads), 0, s, nb, (const uint32_t*)hist, moff,
                       (uint32_t*)nullptr, w.nnz, (int*)nullptr);
    if (rp_type == TG_I64)
        hipLaunchKernelGGL((bk_out_kernel<T, int64_t>), dim3(nb), dim3(256), 0, s, m, P.rows, (const uint32_t*)off,
                           (const uint32_t*)moff, (const uint32_t*)rowoff, (const int32_t*)tci, (const T*)tval,
                           (int64_t*)rp_out, ci_out, val_out, (const int*)(w.bad + 1));
    else
        hipLaunchKernelGGL((bk_out_kernel<T, int32_t>), dim3(nb), dim3(256), 0, s, m, P.rows, (const uint32_t*)off,
                           (const uint32_t*)moff, (const uint32_t*)rowoff, (const int32_t*)tci, (const T*)tval,
                           (int32_t*)rp_out, ci_out, val_out, (const int*)(w.bad + 1));
    TG_LAUNCH_CHECK();
    return triples_found(w, nnz, bad, unfit, s);
}

template <typename T>
static int from_triples_t(int64_t count, const int32_t* I, const int32_t* J, const T* V, int32_t m, int32_t n,
                          int compress, int symmetrize, void* rp_out, tg_dtype rp_type, int32_t* ci_out, T* val_out,
                          int64_t cap, void* ws, size_t ws_bytes, int64_t* nnz_host, hipStream_t s) {
    const int64_t total = symmetrize ? 2 * count : count;
    if (cap < total) return fail(TG_ERR_INVALID, "from_triples: output capacity %lld < %lld", (long long)cap,
                                 (long long)total);
    if (total > (int64_t)0xffffffffll) return fail(TG_ERR_INVALID, "from_triples: too many triples");
    TriplesWs w;
    if (!ws || ws_bytes < triples_ws(count, m, symmetrize, nullptr, nullptr))
        return fail(TG_ERR_WORKSPACE, "from_triples: workspace missing or too small");
    triples_ws(count, m, symmetrize, (char*)ws, &w);
    const BucketPlan P = bucket_plan(total, m, symmetrize ? std::max(m, n) : n);
    if (P.buckets > 0) {
        int64_t nnz = 0;
        int bad = 0, unfit = 0;
        const int rc = bucket_triples<T>(P, count, total, I, J, V, m, n, compress, rp_out, rp_type, ci_out, val_out, w,
                                         &nnz, &bad, &unfit, s);
        if (rc) return rc;
        if (bad) return fail(TG_ERR_INVALID, "from_triples: a row or column index is out of range");
        if (!unfit) {
            if (nnz_host) *nnz_host = nnz;
            return TG_OK;
        }
    }
    hipLaunchKernelGGL(st_zero64_kernel, dim3(grid_of(m + 1)), dim3(256), 0, s, (int64_t)m + 1, w.rowcnt, w.bad);
    if (total > 0) {
        // columns and, for transposed copies, rows appear in either half
        const int cb = bits_of(symmetrize ? std::max(m, n) : n), rb = bits_of((int64_t)(symmetrize ? std::max(m, n) : m) + 1);
        hipLaunchKernelGGL(st_expand_kernel, dim3(grid_of(total)), dim3(256), 0, s, count, I, J, m, n, symmetrize, cb,
                           w.keys[0], w.idx[0], w.bad);
        size_t tb = w.temp_bytes;
        TG_HIP(rocprim::radix_sort_pairs(w.temp, tb, w.keys[0], w.keys[1], w.idx[0], w.idx[1], (size_t)total, 0,
                                         cb + rb, s));
        hipLaunchKernelGGL(st_heads_kernel, dim3(grid_of(total)), dim3(256), 0, s, total, (const uint64_t*)w.keys[1],
                           compress, (uint64_t)(uint32_t)m << cb, w.head);
        tb = w.temp_bytes;
        TG_HIP(rocprim::exclusive_scan(w.temp, tb, (const int64_t*)w.head, w.pos, (int64_t)0, (size_t)total,
                                       rocprim::plus<int64_t>(), s));
        hipLaunchKernelGGL((st_write_kernel<T>), dim3(grid_of(total)), dim3(256), 0, s, total,
                           (const uint64_t*)w.keys[1], (const uint32_t*)w.idx[1], (const int64_t*)w.head,
                           (const int64_t*)w.pos, count, cb, V, compress, ci_out, val_out, w.rowcnt);
    }
    size_t tb = w.temp_bytes;
    TG_HIP(rocprim::exclusive_scan(w.temp, tb, (const int64_t*)w.rowcnt, w.rowscan, (int64_t)0, (size_t)m + 1,
                                   rocprim::plus<int64_t>(), s));
    if (rp_type == TG_I64)
        hipLaunchKernelGGL((st_rp_kernel<int64_t>), dim3(grid_of(m + 1)), dim3(256), 0, s, m,
                           (const int64_t*)w.rowscan, (int64_t*)rp_out, w.nnz);
    else
        hipLaunchKernelGGL((st_rp_kernel<int32_t>), dim3(grid_of(m + 1)), dim3(256), 0, s, m,
                           (const int64_t*)w.rowscan, (int32_t*)rp_out, w.nnz);
    TG_LAUNCH_CHECK();
    int64_t nnz = 0;
    int bad = 0, unfit = 0;
    const int rc = triples_found(w, &nnz, &bad, &unfit, s);
    if (rc) return rc;
    if (bad) return fail(TG_ERR_INVALID, "from_triples: a row or column index is out of range");
    if (rp_type == TG_I32 && nnz > 0x7fffffffll)
        return fail(TG_ERR_DTYPE, "from_triples: nnz does not fit int32 row pointers");
    if (nnz_host) *nnz_host = nnz;
    return TG_OK;
}

// ---- transpose: triples (ci[e], row(e), val[e]) ---------------------------
template <typename RP>
__global__ void st_rows_kernel(int32_t m, const RP* __restrict__ rp, int32_t* __restrict__ rows) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
        for (int64_t e = rp[i]; e < (int64_t)rp[i + 1]; ++e) rows[e] = (int32_t)i;
}

// ---- sparse x sparse expansion ---------------------------------------------
template <typename RP>
__global__ void st_expand_count_kernel(int32_t m, const RP* __restrict__ Arp, const int32_t* __restrict__ Aci,
                                       const RP* __restrict__ Brp, int64_t* __restrict__ cnt) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t c = 0;
        for (int64_t e = Arp[i]; e < (int64_t)Arp[i + 1]; ++e) {
            const int32_t j = Aci[e];
            c += (int64_t)Brp[j + 1] - (int64_t)Brp[j];
        }
        cnt[i] = c;
    }
}

template <typename T, typename RP>
__global__ void st_expand_pairs_kernel(int32_t m, const RP* __restrict__ Arp, const int32_t* __restrict__ Aci,
                                       const T* __restrict__ Aval, const RP* __restrict__ Brp,
                                       const int32_t* __restrict__ Bci, const T* __restrict__ Bval,
                                       const int64_t* __restrict__ off, int32_t* __restrict__ I, int32_t* __restrict__ J,
                                       T* __restrict__ V) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t p = off[i];
        for (int64_t e = Arp[i]; e < (int64_t)Arp[i + 1]; ++e) {
            const int32_t j = Aci[e];
            const T a = Aval ? Aval[e] : T(1);
            for (int64_t f = Brp[j]; f < (int64_t)Brp[j + 1]; ++f, ++p) {
                I[p] = (int32_t)i;
                J[p] = Bci[f];
                if (V) V[p] = a * Bval[f];
            }
        }
    }
}

}  // namespace tg

using namespace tg;

extern "C" size_t tg_csr_from_triples_workspace_bytes(int64_t count, int32_t m, int32_t symmetrize) {
    if (count < 0 || m < 0) return 0;
    return triples_ws(count, m, symmetrize ? 1 : 0, nullptr, nullptr);
}

extern "C" int tg_csr_from_triples(int64_t count, const int32_t* I, const int32_t* J, const void* V,
                                   tg_dtype val_type, int32_t m, int32_t n, int32_t compress, int32_t symmetrize,
                                   void* rp_out, tg_dtype rp_type, int32_t* ci_out, void* val_out, int64_t capacity,
                                   void* workspace, size_t workspace_bytes, int64_t* nnz_out, void* stream) {
    if (nnz_out) *nnz_out = 0;
    if (count < 0 || m < 0 || n < 0 || !rp_out || (count > 0 && (!I || !J || !ci_out)) || (V && !val_out))
        return fail(TG_ERR_INVALID, "tg_csr_from_triples: bad argument");
    if (rp_type != TG_I32 && rp_type != TG_I64) return fail(TG_ERR_DTYPE, "tg_csr_from_triples: rp_type must be I32/I64");
    hipStream_t s = as_stream(stream);
    if (val_type == TG_F64)
        return from_triples_t<double>(count, I, J, (const double*)V, m, n, compress, symmetrize, rp_out, rp_type, ci_out,
                                      (double*)val_out, capacity, workspace, workspace_bytes, nnz_out, s);
    if (val_type == TG_F32)
        return from_triples_t<float>(count, I, J, (const float*)V, m, n, compress, symmetrize, rp_out, rp_type, ci_out,
                                     (float*)val_out, capacity, workspace, workspace_bytes, nnz_out, s);
    return fail(TG_ERR_DTYPE, "tg_csr_from_triples: val_type must be F64/F32");
}

extern "C" size_t tg_csr_transpose_workspace_bytes(int32_t m, int32_t n, int64_t nnz) {
    if (m < 0 || n < 0 || nnz < 0) return 0;
    return align256((size_t)std::max<int64_t>(nnz, 1) * 4) + triples_ws(nnz, n, 0, nullptr, nullptr);
}

extern "C" int tg_csr_transpose(int32_t m, int32_t n, int64_t nnz, const void* rp, tg_dtype rp_type,
                                const int32_t* ci, const void* val, tg_dtype val_type, void* out_rp,
                                int32_t* out_ci, void* out_val, void* workspace, size_t workspace_bytes,
                                void* stream) {
    if (m < 0 || n < 0 || nnz < 0 || !rp || !out_rp || (nnz > 0 && (!ci || !out_ci)) || (val && !out_val))
        return fail(TG_ERR_INVALID, "tg_csr_transpose: bad argument");
    if (!workspace || workspace_bytes < tg_csr_transpose_workspace_bytes(m, n, nnz))
        return fail(TG_ERR_WORKSPACE, "tg_csr_transpose: workspace missing or too small");
    hipStream_t s = as_stream(stream);
    int32_t* rows = (int32_t*)workspace;
    void* rest = (char*)workspace + align256((size_t)std::max<int64_t>(nnz, 1) * 4);
    const size_t rest_bytes = workspace_bytes - align256((size_t)std::max<int64_t>(nnz, 1) * 4);
    if (rp_type == TG_I64)
        hipLaunchKernelGGL((st_rows_kernel<int64_t>), dim3(grid_of(m)), dim3(256), 0, s, m, (const int64_t*)rp, rows);
    else if (rp_type == TG_I32)
        hipLaunchKernelGGL((st_rows_kernel<int32_t>), dim3(grid_of(m)), dim3(256), 0, s, m, (const int32_t*)rp, rows);
    else
        return fail(TG_ERR_DTYPE, "tg_csr_transpose: rp_type must be I32/I64");
    TG_LAUNCH_CHECK();
    int64_t got = 0;
    // (i, j, a) of A becomes (j, i, a): rows of A^T are the columns of A
    int rc;
    if (val_type == TG_F32)
        rc = from_triples_t<float>(nnz, ci, rows, (const float*)val, n, m, 0, 0, out_rp, rp_type, out_ci,
                                   (float*)out_val, nnz, rest, rest_bytes, &got, s);
    else
        rc = from_triples_t<double>(nnz, ci, rows, (const double*)val, n, m, 0, 0, out_rp, rp_type, out_ci,
                                    (double*)out_val, nnz, rest, rest_bytes, &got, s);
    return rc;
}

// Expanded (pre-compression) nonzero count of A * B; synchronises `stream`.
extern "C" int tg_csr_spgemm_expanded_count(int32_t m, const void* Arp, const int32_t* Aci, const void* Brp,
                                            tg_dtype rp_type, int64_t* count_out, void* workspace,
                                            size_t workspace_bytes, void* stream) {
    if (m < 0 || !Arp || !Brp || !count_out) return fail(TG_ERR_INVALID, "tg_csr_spgemm_expanded_count: bad argument");
    size_t scan_tmp = 0;
    (void)rocprim::exclusive_scan(nullptr, scan_tmp, (const int64_t*)nullptr, (int64_t*)nullptr, (int64_t)0, (size_t)m + 1,
                            rocprim::plus<int64_t>());
    const size_t need = 2 * align256(8 * ((size_t)m + 1)) + align256(scan_tmp);
    if (!workspace || workspace_bytes < need)
        return fail(TG_ERR_WORKSPACE, "tg_csr_spgemm_expanded_count: workspace must hold %zu bytes", need);
    hipStream_t s = as_stream(stream);
    int64_t* cnt = (int64_t*)workspace;
    int64_t* off = (int64_t*)((char*)workspace + align256(8 * ((size_t)m + 1)));
    void* tmp = (char*)workspace + 2 * align256(8 * ((size_t)m + 1));
    hipLaunchKernelGGL(st_zero64_kernel, dim3(grid_of(m + 1)), dim3(256), 0, s, (int64_t)m + 1, cnt);
    if (rp_type == TG_I64)
        hipLaunchKernelGGL((st_expand_count_kernel<int64_t>), dim3(grid_of(m)), dim3(256), 0, s, m, (const int64_t*)Arp,
                           Aci, (const int64_t*)Brp, cnt);
    else
        hipLaunchKernelGGL((st_expand_count_kernel<int32_t>), dim3(grid_of(m)), dim3(256), 0, s, m, (const int32_t*)Arp,
                           Aci, (const int32_t*)Brp, cnt);
    TG_LAUNCH_CHECK();
    TG_HIP(rocprim::exclusive_scan(tmp, scan_tmp, (const int64_t*)cnt, off, (int64_t)0, (size_t)m + 1,
                                   rocprim::plus<int64_t>(), s));
    TG_HIP(hipMemcpyAsync(count_out, off + m, 8, hipMemcpyDeviceToHost, s));
    TG_HIP(hipStreamSynchronize(s));
    return TG_OK;
}

extern "C" size_t tg_csr_spgemm_workspace_bytes(int32_t m, int32_t n, int64_t expanded, tg_dtype val_type) {
    size_t scan_tmp = 0;
    (void)rocprim::exclusive_scan(nullptr, scan_tmp, (const int64_t*)nullptr, (int64_t*)nullptr, (int64_t)0, (size_t)m + 1,
                            rocprim::plus<int64_t>());
    const size_t vs = val_type == TG_F32 ? 4 : 8;
    return 2 * align256(8 * ((size_t)m + 1)) + align256(scan_tmp) + 2 * align256(4 * (size_t)std::max<int64_t>(expanded, 1)) +
           align256(vs * (size_t)std::max<int64_t>(expanded, 1)) + triples_ws(expanded, m, 0, nullptr, nullptr);
}

// C = A * B (A: m x k, B: k x n).  Outputs need capacity `expanded` (from
// tg_csr_spgemm_expanded_count); *nnz_out receives the compressed count.
// Values null on both A and B -> pattern product (DotBinary_).
extern "C" int tg_csr_spgemm(int32_t m, int32_t k, int32_t n, const void* Arp, const int32_t* Aci, const void* Aval,
                             const void* Brp, const int32_t* Bci, const void* Bval, tg_dtype rp_type,
                             tg_dtype val_type, int64_t expanded, void* Crp, int32_t* Cci, void* Cval,
                             void* workspace, size_t workspace_bytes, int64_t* nnz_out, void* stream) {
    if (m < 0 || k < 0 || n < 0 || expanded < 0 || !Arp || !Brp || !Crp || ((Aval == nullptr) != (Bval == nullptr)))
        return fail(TG_ERR_INVALID, "tg_csr_spgemm: bad argument");
    if (!workspace || workspace_bytes < tg_csr_spgemm_workspace_bytes(m, n, expanded, val_type))
        return fail(TG_ERR_WORKSPACE, "tg_csr_spgemm: workspace missing or too small");
    hipStream_t s = as_stream(stream);
    size_t scan_tmp = 0;
    (void)rocprim::exclusive_scan(nullptr, scan_tmp, (const int64_t*)nullptr, (int64_t*)nullptr, (int64_t)0, (size_t)m + 1,
                            rocprim::plus<int64_t>());
    char* w = (char*)workspace;
    int64_t* cnt = (int64_t*)w;
    w += align256(8 * ((size_t)m + 1));
    int64_t* off = (int64_t*)w;
    w += align256(8 * ((size_t)m + 1));
    void* tmp = w;
    w += align256(scan_tmp);
    const size_t E = (size_t)std::max<int64_t>(expanded, 1);
    int32_t* I = (int32_t*)w;
    w += align256(4 * E);
    int32_t* J = (int32_t*)w;
    w += align256(4 * E);
    void* V = w;
    w += align256((val_type == TG_F32 ? 4 : 8) * E);
    const size_t rest_bytes = workspace_bytes - (size_t)(w - (char*)workspace);
    hipLaunchKernelGGL(st_zero64_kernel, dim3(grid_of(m + 1)), dim3(256), 0, s, (int64_t)m + 1, cnt);
    const bool i64 = rp_type == TG_I64;
    if (i64)
        hipLaunchKernelGGL((st_expand_count_kernel<int64_t>), dim3(grid_of(m)), dim3(256), 0, s, m, (const int64_t*)Arp,
                           Aci, (const int64_t*)Brp, cnt);
    else
        hipLaunchKernelGGL((st_expand_count_kernel<int32_t>), dim3(grid_of(m)), dim3(256), 0, s, m, (const int32_t*)Arp,
                           Aci, (const int32_t*)Brp, cnt);
    TG_HIP(rocprim::exclusive_scan(tmp, scan_tmp, (const int64_t*)cnt, off, (int64_t)0, (size_t)m + 1,
                                   rocprim::plus<int64_t>(), s));
    const bool vals = Aval != nullptr;
#define TG_EXPAND(TT, RPT)                                                                                          \
    hipLaunchKernelGGL((st_expand_pairs_kernel<TT, RPT>), dim3(grid_of(m)), dim3(256), 0, s, m, (const RPT*)Arp, Aci, \
                       (const TT*)Aval, (const RPT*)Brp, Bci, (const TT*)Bval, (const int64_t*)off, I, J,             \
                       vals ? (TT*)V : (TT*)nullptr)
    if (val_type == TG_F32) {
        if (i64) TG_EXPAND(float, int64_t); else TG_EXPAND(float, int32_t);
    } else {
        if (i64) TG_EXPAND(double, int64_t); else TG_EXPAND(double, int32_t);
    }
#undef TG_EXPAND
    TG_LAUNCH_CHECK();
    if (val_type == TG_F32)
        return from_triples_t<float>(expanded, I, J, vals ? (const float*)V : nullptr, m, n, 1, 0, Crp, rp_type, Cci,
                                     (float*)Cval, expanded, w, rest_bytes, nnz_out, s);
    return from_triples_t<double>(expanded, I, J, vals ? (const double*)V : nullptr, m, n, 1, 0, Crp, rp_type, Cci,
                                  (double*)Cval, expanded, w, rest_bytes, nnz_out, s);
}
