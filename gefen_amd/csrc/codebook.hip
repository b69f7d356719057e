// Codebook learning on the device: lookup tables for the nearest-codeword
// search, the block-normalised 4096-bin histogram, the exact-DP quantiser and
// the Lloyd-Max accumulators.
//
// Histogram: gefen.py:350-366.  Exact DP: quantization.py:206-258 with the
// histogram statistics of gefen.py:373-399; the DP is evaluated level by level
// (one launch per cluster count), one wave per segment end, over the starts that
// a bound on the cost leaves, with the reference's strict "<" (first best start
// wins) reproduced by a lexicographic (cost, start) minimum.  All float64 arithmetic is written without
// contraction, so every cost and codeword equals the reference's.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "capi_internal.h"
#include "common.h"

namespace gefen {

// ---------------------------------------------------------------------------
// codebook tables (see CodebookTables in common.h)
__device__ __forceinline__ int32_t f_ord(float x) {
    const uint32_t b = __float_as_uint(x);
    return (b & 0x80000000u) ? -(int32_t)(b & 0x7fffffffu) : (int32_t)b;
}
__device__ __forceinline__ float f_dec(int32_t o) {
    return o >= 0 ? __uint_as_float((uint32_t)o) : __uint_as_float(0x80000000u | (uint32_t)(-o));
}

// byte offsets of the fields the GPU tests read from a prepared table
static_assert(offsetof(CodebookTables, bucket_fine) == 6176 && offsetof(CodebookTables, max_probe) == 22588 &&
                  offsetof(CodebookTables, max_probe_fine) == 22592 && offsetof(CodebookTables, nb16) == 22608,
              "codebook table layout");

// #{k in [1, K) : thr[k] < x} by bisection, in the same eight steps for every x, so
// that a thread's searches overlap.
__device__ __forceinline__ int thresholds_below(const float* thr, int K, float x) {
    int lo = 1, hi = K;  // first k in [1, K) with thr[k] >= x
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int mid = (lo + hi) >> 1;  // <= 256
        const bool open = lo < hi, less = thr[mid] < x;
        lo = open && less ? mid + 1 : lo;
        hi = open && !less ? mid : hi;
    }
    return lo - 1;
}

// One workgroup, as max_probe needs all cells.  Bound by the latency of the searches
// (eight dependent LDS reads each): one after another in 256 threads 42 us; 1024
// threads with their searches interleaved 11.
constexpr int kPrepThreads = 1024;
__global__ __launch_bounds__(kPrepThreads) void k_prepare_codebook(const float* __restrict__ cb, int K,
                                                                   CodebookTables* __restrict__ T) {
    __shared__ float thr[260];
    __shared__ uint16_t bk[kFineCells + 1];
    __shared__ int probe_max, probe_max_fine;
    const int t = threadIdx.x;
    if (t < 256) T->cb[t] = t < K ? cb[t] : __builtin_inff();
    if (t == 0) T->K = K;
    // thr[k], k = 1..K-1: largest x in (cb[k-1], cb[k]] where the left entry wins
    for (int k = t; k < 260; k += kPrepThreads) {
        float v = __builtin_inff();
        if (k >= 1 && k < K) {
            const float a = cb[k - 1], b = cb[k];
            if (!(b > a)) {
                v = a;
            } else {
                int32_t lo = f_ord(a), hi = f_ord(b);  // pred(lo) holds (or lo is a), pred(hi) fails
                while (hi - lo > 1) {
                    const int32_t mid = lo + (hi - lo) / 2;
                    const float x = f_dec(mid);
                    if (fabsf(x - a) <= fabsf(x - b)) lo = mid; else hi = mid;
                }
                v = f_dec(lo);
            }
        } else if (k == 0) {
            v = -__builtin_inff();
        }
        thr[k] = v;
        T->thr[k] = v;
    }
    __syncthreads();
    // bucket_fine[e] = #{k in 1..K-1 : thr[k] < -1 + e/4096}; bucket[e] = bucket8[e] = bucket_fine[2e]
#pragma unroll
    for (int r = 0; r <= kFineCells / kPrepThreads; ++r) {
        const int e = t + r * kPrepThreads;
        const float edge = -1.0f + (float)e * 0.000244140625f;  // exact: a multiple of 2^-12
        const uint16_t c = (uint16_t)thresholds_below(thr, K, edge);
        if (e > kFineCells) continue;
        T->bucket_fine[e] = (uint8_t)c;  // c <= K - 1 <= 255
        if (!(e & 1)) {
            T->bucket[e >> 1] = c;
            T->bucket8[e >> 1] = (uint8_t)c;
        }
        bk[e] = c;
    }
    for (int e = kFineCells + 1 + t; e < kFineBytes; e += kPrepThreads) T->bucket_fine[e] = 0;
    if (t < kBucket8Bytes - 4097) T->bucket8[4097 + t] = 0;
    if (t < 3) T->bucket[4097 + t] = 0;
    if (t == 0) probe_max = probe_max_fine = 0;
    __syncthreads();
    // a search from bucket b (one below x's bucket) meets the thresholds in
    // [edge_b, edge_b+2); past the last edges it meets every finite one left
    int worst = 0, worst_fine = 0;
    for (int b = t; b <= kFineCells; b += kPrepThreads) {
        const int hi = (b + 2 <= kFineCells) ? (int)bk[b + 2] : (K - 1);
        const int n = hi - (int)bk[b];
        worst_fine = n > worst_fine ? n : worst_fine;
        if (!(b & 1)) {
            const int hc = (b + 4 <= kFineCells) ? (int)bk[b + 4] : (K - 1);
            const int nc = hc - (int)bk[b];
            worst = nc > worst ? nc : worst;
        }
    }
    worst = (int)wave_group_max_u32((uint32_t)worst, 64);  // counts: non-negative where thr is sorted
    worst_fine = (int)wave_group_max_u32((uint32_t)worst_fine, 64);
    if ((t & 63) == 0) {
        atomicMax(&probe_max, worst);
        atomicMax(&probe_max_fine, worst_fine);
    }
    __syncthreads();
    if (t == 0) {
        T->max_probe = (bk[0] != 0) ? 1 << 20 : probe_max;
        T->max_probe_fine = (bk[0] != 0) ? 1 << 20 : probe_max_fine;
    }
    // nb16: #{k in 1..K-1 : thr[k] < x} for the bf16 values x of the table
#pragma unroll
    for (int r = 0; r < (kNb16Bytes + kPrepThreads - 1) / kPrepThreads; ++r) {
        const int i = t + r * kPrepThreads;
        const uint32_t bits = i >= (int)kNb16Side ? kNb16Lo + (uint32_t)(i - (int)kNb16Side)
                                                  : 0x8000u | (kNb16Lo + kNb16Side - 1u - (uint32_t)i);
        const uint8_t c = (uint8_t)thresholds_below(thr, K, __uint_as_float(bits << 16));
        if (i < kNb16Bytes) T->nb16[i] = i < 2 * (int)kNb16Side ? c : 0;
    }
}

// ---------------------------------------------------------------------------
// histogram: a lane group per block row, LDS-privatised counts per workgroup, many
// tensors per launch.
constexpr int kHistTasks = 56;
constexpr int kHistBins = 4096;
constexpr int kHistMaxWgs = 1024;  // of one tensor
struct HistTask {
    const void* g;
    unsigned long long* counts;
    int64_t nrows;
    int64_t rowlen;
    int32_t nvec;      // vectors of W elements per row, the last one shifted back to end with the row
    int32_t lpr_log2;  // lanes per row
};
struct HistBatch {
    HistTask t[kHistTasks];
    int32_t wg_begin[kHistTasks + 1];
    int32_t ntasks;
    int32_t bins;
    int32_t pow2;      // bins is a power of two: dividing by the bin width is exact scaling by its reciprocal
    float bw, scale;
};
static_assert(sizeof(HistBatch) <= 4000, "kernel arguments are limited to 4 KB");

// clamp(floor((x + 1) / bw), 0, bins - 1), NaN -> 0 (its conversion to int64 is INT64_MIN)
__device__ __forceinline__ int hist_bin(float x, const HistBatch& B) {
    const float y = B.pow2 ? (x + 1.0f) * B.scale : (x + 1.0f) / B.bw;
    return (int)fminf(fmaxf(y, 0.0f), (float)(B.bins - 1));
}

// A row's maximum as its elements are divided by it.  The quotient is Markstein's:
// q = v * (1 / amax), x = q + (v - q amax) (1 / amax), which is the IEEE quotient
// when 1 / amax is rounded correctly and v - q amax is exact; with amax >= 2^-60 that
// holds for every v above 2^-86 (the subnormal bits reach 2^-149), and a smaller v
// has |x| < 2^-26, whose bin does not depend on its last bits (x + 1 = 1).
struct RowMax {
    float amax, inv;
    bool fast, positive;
    __device__ __forceinline__ explicit RowMax(float m) : amax(m), inv(1.0f / m) {
        fast = m >= 0x1p-60f && m <= 0x1p120f;
        positive = m > 0.0f;  // NaN and zero maxima normalise to zero
    }
    __device__ __forceinline__ float divide(float v) const {
        if (fast) {
            const float q = v * inv;
            return __builtin_fmaf(__builtin_fmaf(-q, amax, v), inv, q);
        }
        return positive ? v / amax : 0.0f;
    }
};

__device__ __forceinline__ int hist_task(const HistBatch& B) {
    int lo = 0, hi = B.ntasks - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (B.wg_begin[mid] <= (int)blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Rows of up to lanes * W * R elements, held in registers: read once, 16 bytes per
// lane at any alignment.  R = 0: longer rows, a wave each, read twice.  Bound by
// the LDS atomics and the instructions around them (about a dozen per element).
// 64M float32 values in rows of 2048: 65 us (two reads and an IEEE division: 151).
template <typename T, int W, int R>
__global__ __launch_bounds__(256) void k_histogram(const HistBatch B) {
    __shared__ uint32_t h[kHistBins];
    for (int i = threadIdx.x; i < B.bins; i += 256) h[i] = 0;
    __syncthreads();
    const int ti = hist_task(B);
    const HistTask K = B.t[ti];
    const T* __restrict__ g = static_cast<const T*>(K.g);
    const int lane = threadIdx.x & 63;
    const int nwg = B.wg_begin[ti + 1] - B.wg_begin[ti];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t first = ((int64_t)blockIdx.x - B.wg_begin[ti]) * 4 + wave, step = (int64_t)nwg * 4;
    if constexpr (R > 0) {
        const int lpr = 1 << K.lpr_log2, lir = lane & (lpr - 1);
        const int rpw = 64 >> K.lpr_log2;
        const int64_t units = (K.nrows + rpw - 1) / rpw;
        for (int64_t unit = first; unit < units; unit += step) {
            const int64_t row = unit * rpw + (lane >> K.lpr_log2);
            const bool active = row < K.nrows;
            const T* __restrict__ src = g + (active ? row : K.nrows - 1) * K.rowlen;
            AnyVec<T, W> v[R];
            uint32_t key = 0;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                const int64_t e = min((int64_t)min(lir + j * lpr, K.nvec - 1) * W, K.rowlen - W);
                v[j] = *reinterpret_cast<const AnyVec<T, W>*>(src + e);
            }
#pragma unroll
            for (int j = 0; j < R; ++j)
#pragma unroll
                for (int w = 0; w < W; ++w) key = max(key, abs_key(to_f32(v[j].v[w])));
            const RowMax M(__uint_as_float(wave_group_max_u32(key, lpr)));
            if (!active) continue;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                const int q = lir + j * lpr;
                if (q >= K.nvec) continue;
                // elements of the last vector that the one before it has counted
                const int skip = (int)max((int64_t)(q + 1) * W - K.rowlen, (int64_t)0);
#pragma unroll
                for (int w = 0; w < W; ++w)
                    if (w >= skip) atomicAdd(&h[hist_bin(M.divide(to_f32(v[j].v[w])), B)], 1u);
            }
        }
    } else {
        for (int64_t row = first; row < K.nrows; row += step) {
            const T* __restrict__ src = g + row * K.rowlen;
            uint32_t key = 0;
            for (int64_t j = lane; j < K.rowlen; j += 64) key = max(key, abs_key(to_f32(src[j])));
            const RowMax M(__uint_as_float(wave_group_max_u32(key, 64)));
            for (int64_t j = lane; j < K.rowlen; j += 64) atomicAdd(&h[hist_bin(M.divide(to_f32(src[j])), B)], 1u);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < B.bins; i += 256)
        if (h[i]) atomicAdd(&K.counts[i], (unsigned long long)h[i]);
}

// Rows of one element: x = v / |v| is -1, 1, 0 for a zero (or a NaN, whose maximum is
// not positive) or NaN for an infinity: three bins, counted in registers (in LDS all
// lanes' atomics would meet in two addresses).
template <typename T, int W>
__global__ __launch_bounds__(256) void k_histogram_signs(const HistBatch B) {
    __shared__ uint32_t red[4][4];
    const int ti = hist_task(B);
    const HistTask K = B.t[ti];
    const T* __restrict__ g = static_cast<const T*>(K.g);
    const int64_t nwg = B.wg_begin[ti + 1] - B.wg_begin[ti];
    const int64_t me = ((int64_t)blockIdx.x - B.wg_begin[ti]) * 256 + threadIdx.x;
    uint32_t neg = 0, pos = 0, inf = 0, all = 0;
    auto count = [&](float v) {
        const uint32_t b = __float_as_uint(v), m = b & 0x7fffffffu;
        const bool finite = m - 1u < 0x7f7fffffu;  // not zero, infinite or NaN
        neg += finite && (b >> 31) ? 1u : 0u;
        pos += finite && !(b >> 31) ? 1u : 0u;
        inf += m == 0x7f800000u ? 1u : 0u;
    };
    const int64_t whole = K.nrows / W;
    for (int64_t q = me; q < whole; q += nwg * 256) {
        const AnyVec<T, W> v = *reinterpret_cast<const AnyVec<T, W>*>(g + q * W);
#pragma unroll
        for (int w = 0; w < W; ++w) count(to_f32(v.v[w]));
        all += W;
    }
    if (me < K.nrows - whole * W) {
        count(to_f32(g[whole * W + me]));
        all += 1;
    }
    uint32_t c[4] = {neg, pos, inf, all};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        for (int off = 32; off > 0; off >>= 1) c[k] += (uint32_t)__shfl_xor((int)c[k], off, 64);
        if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = c[k];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        auto total = [&](int k) { return (red[k][0] + red[k][1]) + (red[k][2] + red[k][3]); };
        const uint32_t n = total(0), p = total(1), i = total(2), a = total(3);
        const uint32_t mine = threadIdx.x == 0 ? n : threadIdx.x == 1 ? p : threadIdx.x == 2 ? i : a - n - p - i;
        const float x = threadIdx.x == 0 ? -1.0f : threadIdx.x == 1 ? 1.0f : threadIdx.x == 2 ? __builtin_nanf("") : 0.0f;
        if (mine) atomicAdd(&K.counts[hist_bin(x, B)], (unsigned long long)mine);
    }
}

// acc[b] += float(counts[t][b]) for the tasks in order (gefen.py:331, 347, 365 sum in float32)
__global__ __launch_bounds__(64) void k_accumulate_tasks(float* __restrict__ acc, const int64_t* __restrict__ counts,
                                                         int ntasks, int bins) {
    const int b = blockIdx.x * 64 + threadIdx.x;
    if (b >= bins) return;
    float a = acc[b];
    int t = 0;
    for (; t + 16 <= ntasks; t += 16) {
        float c[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) c[u] = (float)counts[(int64_t)(t + u) * bins + b];
#pragma unroll
        for (int u = 0; u < 16; ++u) a = a + c[u];
    }
    for (; t < ntasks; ++t) a = a + (float)counts[(int64_t)t * bins + b];
    acc[b] = a;
}

__global__ __launch_bounds__(256) void k_zero_i64(int64_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_accumulate_counts(float* __restrict__ acc, const int64_t* __restrict__ counts, int bins) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < bins) acc[i] = acc[i] + (float)counts[i];
}

// ---------------------------------------------------------------------------
// exact DP workspace:
//   header  int32[64]      : [0] N active bins, [1] status (0 ok, 1 padded done, 2 empty),
//                            [2..3] the cut's slack as a double (dp_slack)
//   pw, pwx, pwx2          : double[bins + 1] each (prefix sums, sequential order)
//   dp                     : double[(K + 1) * (bins + 1)], level-major
//   bt                     : int32[(K + 1) * (bins + 1)]
//   jump                   : int32[kDpGroups * (bins + 1)], see k_dp_jump
//   cw                     : float[bins] active centres
constexpr int kDpMaxK = 256;
constexpr int kDpGroup = 16;  // levels that one jump table crosses
constexpr int kDpGroups = kDpMaxK / kDpGroup;
struct DpLayout {
    size_t pw, pwx, pwx2, dp, bt, jump, cw, total;
    DpLayout(int bins, int K) {
        size_t o = 256;
        pw = o;  o += sizeof(double) * (bins + 1);
        pwx = o; o += sizeof(double) * (bins + 1);
        pwx2 = o; o += sizeof(double) * (bins + 1);
        dp = o;  o += sizeof(double) * (size_t)(K + 1) * (bins + 1);
        bt = o;  o += sizeof(int32_t) * (size_t)(K + 1) * (bins + 1);
        jump = o; o += sizeof(int32_t) * (size_t)kDpGroups * (bins + 1);
        cw = o;  o += sizeof(float) * bins;
        total = o;
    }
};

constexpr int kDpMaxBins = 4096;
constexpr int kDpInitThreads = 256;

// How much a segment's cost alone may exceed the best candidate before longer segments
// are left out (k_dp_level), for counts of this sum W and smallest value m; infinite,
// which leaves nothing out, where no such bound holds.  In exact arithmetic a segment's
// cost never falls when it grows, and dp >= 0.  In float64 a prefix sum of up to 4096
// counts is within 2^-41 W of the exact one (|x| < 1), so a segment's sums sw, swx and
// swx2 are within h = 2^-40 W of theirs.  The error of swx^2 / sw is then at most
// h (3 sw + h) / (sw - h), 4 h where sw >= m >= 5 h, a cost's 5 h < 2^-37 W and a dp
// value's (up to 256 costs) 2^-29 W: 2^-28 W covers both with room, and is far below the
// costs it is compared with (5e-6 W for 256 even levels).  Where m < 5 h the divisor can
// cancel, and a cost be off by any amount: counts that span about 15 decades and more gave
// another codebook than the full search.  2^37 below is 2^40 / 5 rounded down; an
// optimizer's counts, whole numbers, exceed it only past 1.4e11 elements.  256 codewords
// of 4096 full bins: 1.7 ms with the bound, 6.5 without.
__device__ __forceinline__ double dp_slack(double W, double m) {
    return W <= 0x1p37 * m ? 0x1p-28 * W : __builtin_inf();
}

// The first `n` values of v (LDS, n <= kDpMaxK) in ascending order, equal ones as
// they stood (an insertion sort; in parallel it is only checked, since codewords
// come out sorted), written to out.  Every thread of the workgroup takes part.
__device__ __forceinline__ void sort_codewords(float* v, int n, float* __restrict__ out, int* unsorted) {
    const int t = threadIdx.x;
    if (t == 0) *unsorted = 0;
    __syncthreads();
    if (t > 0 && t < n && !(v[t - 1] <= v[t])) *unsorted = 1;
    __syncthreads();
    if (*unsorted && t == 0) {
        for (int i = 1; i < n; ++i) {
            const float x = v[i];
            int j = i - 1;
            while (j >= 0 && v[j] > x) { v[j + 1] = v[j]; --j; }
            v[j + 1] = x;
        }
    }
    __syncthreads();
    if (t < n) out[t] = v[t];
}

// Active bins (count > 0) in bin order, their centres -1 + (2b+1)/bins (exact
// for power-of-two bins), and the float64 prefix sums of w, w x, w x^2
// (torch.cumsum on the CPU, quantization.py:226-231: the element products in
// parallel, then the sums in sequential order).  The workgroup compacts the
// active bins into LDS (a scan of per-thread counts); then one lane of each of
// three waves runs one of the sums in order, the next 32 elements read while the
// current ones are added: a chain of 4096 dependent additions, 18 ns each (one
// lane for all three sums, 16 elements at a time: 132 us; now 76).
__global__ __launch_bounds__(kDpInitThreads) void k_dp_init(const float* __restrict__ counts, int bins, int K,
                                                            int force, char* __restrict__ ws, DpLayout L,
                                                            float* __restrict__ out) {
    constexpr int kPer = kDpMaxBins / kDpInitThreads;  // bins per thread
    __shared__ __attribute__((aligned(16))) double sums[3][kDpMaxBins];
    __shared__ int wave_total[kDpInitThreads / 64];
    __shared__ float wave_least[kDpInitThreads / 64];
    __shared__ float sorted[kDpMaxK];
    __shared__ int unsorted;
    int32_t* hdr = reinterpret_cast<int32_t*>(ws);
    double* pw = reinterpret_cast<double*>(ws + L.pw);
    double* pwx = reinterpret_cast<double*>(ws + L.pwx);
    double* pwx2 = reinterpret_cast<double*>(ws + L.pwx2);
    double* dp = reinterpret_cast<double*>(ws + L.dp);
    float* cw = reinterpret_cast<float*>(ws + L.cw);
    const int t = threadIdx.x, lane = t & 63;
    const int b0 = t * kPer;  // this thread's bins b0 .. b0 + kPer - 1 (in order)
    float mine[kPer], least = __builtin_inff();
    int cnt = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        mine[k] = b0 + k < bins ? counts[b0 + k] : 0.0f;
        cnt += mine[k] > 0.0f ? 1 : 0;
        if (mine[k] > 0.0f) least = fminf(least, mine[k]);
    }
    for (int off = 32; off > 0; off >>= 1) least = fminf(least, __shfl_xor(least, off, 64));
    if (lane == 0) wave_least[t >> 6] = least;
    int incl = cnt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    if (lane == 63) wave_total[t >> 6] = incl;
    __syncthreads();
    int n = incl - cnt, N = 0;
    for (int w = 0; w < kDpInitThreads / 64; ++w) {
        if (w < (t >> 6)) n += wave_total[w];
        N += wave_total[w];
    }
    const double inv_bins = 1.0 / (double)bins;  // exact: bins is a power of two
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        if (mine[k] > 0.0f) {
            const float center = (float)(-1.0 + (2.0 * (b0 + k) + 1.0) * inv_bins);
            const double w = (double)mine[k], x = (double)center;
            sums[0][n] = w;
            sums[1][n] = w * x;
            sums[2][n] = w * (x * x);
            cw[n] = center;
            ++n;
        }
    }
    __syncthreads();
    if (lane == 0 && (t >> 6) < 3) {  // one running sum each, in bin order, in place
        constexpr int kB = 32;
        double* v = sums[t >> 6];
        double a = 0.0, x[kB], y[kB];
        const int whole = N / (2 * kB) * (2 * kB);
        auto read = [&](double* r, int i) {
#pragma unroll
            for (int u = 0; u < kB; ++u) r[u] = v[i + u];
        };
        auto add = [&](double* r, int i) {
#pragma unroll
            for (int u = 0; u < kB; ++u) {
                a = a + r[u];
                r[u] = a;
            }
#pragma unroll
            for (int u = 0; u < kB; ++u) v[i + u] = r[u];
        };
        if (whole) read(x, 0);
        for (int i = 0; i < whole; i += 2 * kB) {
            read(y, i + kB);
            add(x, i);
            if (i + 2 * kB < whole) read(x, i + 2 * kB);
            add(y, i + kB);
        }
        for (int i = whole; i < N; ++i) {
            a = a + v[i];
            v[i] = a;
        }
    }
    __syncthreads();
    for (int i = t; i <= N; i += kDpInitThreads) {
        pw[i] = i ? sums[0][i - 1] : 0.0;
        pwx[i] = i ? sums[1][i - 1] : 0.0;
        pwx2[i] = i ? sums[2][i - 1] : 0.0;
    }
    if (N > 0 && K <= N)  // dp[0][e]: no segmentation of e > 0 points into zero clusters
        for (int e = t; e <= N; e += kDpInitThreads) dp[e] = e ? __builtin_inf() : 0.0;
    if (N > 0 && K > N) {  // quantization.py:68-81 padded codebook
        if (t < K) sorted[t] = cw[t < N ? t : N - 1];
        if (force && t == 0) sorted[0] = -1.0f;
        if (force && t == K - 1) sorted[K - 1] = 1.0f;
        __syncthreads();
        sort_codewords(sorted, K, out, &unsorted);
    }
    if (t == 0) {
        hdr[0] = N;
        hdr[1] = N == 0 ? 2 : (K > N ? 1 : 0);
        for (int w = 1; w < kDpInitThreads / 64; ++w) least = fminf(least, wave_least[w]);
        *reinterpret_cast<double*>(hdr + 2) = N ? dp_slack(sums[0][N - 1], (double)least) : 0.0;
    }
}
static_assert(kDpMaxBins % kDpInitThreads == 0, "whole bins per thread");
static_assert(kDpInitThreads >= kDpMaxK && kDpInitThreads / 64 >= 3, "one codeword per thread, a wave per sum");

// One DP level (quantization.py:158-186): for every segment end e in [c, N],
// the first start s in [c, e] minimising dp[c-1][s-1] + cost(s, e), in
// float64 with the reference's expression order; strict < keeps the first
// minimum, and the cross-lane reduction takes the lexicographic (cost, start)
// minimum.
//
// A wave takes one end and looks at the starts from the nearest one down, 128 at
// a time, until the cost of the segment alone exceeds the best candidate by the
// slack: then no start further down can be as good (dp_slack).
//
// The optimal segment spans about N / c points, and the bound cuts at N / c^(2/3),
// so most levels are one or two passes per end, bound by the launch and one trip to
// memory.  256 codewords from 4096 full bins: 3.95 -> 1.71 ms (every start of every
// end, from copies of the prefix sums in LDS: 14.7 us a level; now 6.3).
constexpr int kDpThreads = 256;
constexpr int kDpWaves = kDpThreads / 64;
constexpr int kDpUnroll = 2;  // independent candidates per lane and pass (4: 2% slower over all levels)

// Segment cost of starts s (prefix index i = s - 1) for end e: MODE 0 the
// free-centre cost sum_wx2 - sum_wx^2 / sum_w, MODE -1 / +1 the cost about
// the fixed centre -1 / +1 (force_endpoints, first / last cluster).
template <int MODE>
__device__ __forceinline__ double dp_cost(double sw, double swx, double swx2) {
    if (MODE == 0) {
        const double sq = swx * swx;
        return swx2 - sq / sw;
    }
    const double fc = (double)MODE;
    const double t1 = (2.0 * fc) * swx;
    const double t2 = (fc * fc) * sw;
    return (swx2 - t1) + t2;
}

template <int OFF>
__device__ __forceinline__ double min_xor(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint64_t o = ((uint64_t)lane_xor<OFF>((uint32_t)(b >> 32)) << 32) | lane_xor<OFF>((uint32_t)b);
    const double w = __builtin_bit_cast(double, o);
    return w < v ? w : v;
}
__device__ __forceinline__ double wave_min_f64(double v) {
    v = min_xor<1>(v);
    v = min_xor<2>(v);
    v = min_xor<4>(v);
    v = min_xor<8>(v);
    v = min_xor<16>(v);
    return min_xor<32>(v);
}

// The operands of one pass: starts top - lane - 64 u (prefix indices), not below lo.
struct DpPass {
    double p[kDpUnroll], px[kDpUnroll], px2[kDpUnroll], prev[kDpUnroll];
};
struct DpArrays {
    const double *__restrict__ pw, *__restrict__ pwx, *__restrict__ pwx2, *__restrict__ prev;
};
__device__ __forceinline__ DpPass dp_load(const DpArrays& A, int top, int lo, int lane) {
    DpPass r;
#pragma unroll
    for (int u = 0; u < kDpUnroll; ++u) {
        const int i = max(top - lane - 64 * u, lo);
        r.p[u] = A.pw[i];
        r.px[u] = A.pwx[i];
        r.px2[u] = A.pwx2[i];
        r.prev[u] = A.prev[i];
    }
    return r;
}

template <int MODE>
__device__ __forceinline__ void dp_end(DpPass d, double Pe, double PXe, double PX2e, double slack, int top, int lo,
                                       int lane, const DpArrays& A, double* dp_out, int32_t* bt_out) {
    double best = __builtin_inf(), least;
    int bi = -1;  // prefix index s - 1 of the best start
    for (;;) {
        double seg = 0.0;
#pragma unroll
        for (int u = 0; u < kDpUnroll; ++u) {
            const int i = max(top - lane - 64 * u, lo);
            seg = dp_cost<MODE>(Pe - d.p[u], PXe - d.px[u], PX2e - d.px2[u]);
            const double cand = d.prev[u] + seg;
            if (cand < best || (cand == best && bi >= 0 && i < bi)) { best = cand; bi = i; }
        }
        least = wave_min_f64(best);
        // lane 63's last start is the lowest of this pass
        const uint64_t bits = __builtin_bit_cast(uint64_t, seg);
        const uint64_t low = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(bits >> 32), 63) << 32) |
                             (uint32_t)__builtin_amdgcn_readlane((int)bits, 63);
        top -= 64 * kDpUnroll;
        if (top < lo || __builtin_bit_cast(double, low) > least + slack) break;
        d = dp_load(A, top, lo, lane);
    }
    const bool mine = bi >= 0 && best == least;
    const uint64_t who = __builtin_amdgcn_ballot_w64(mine);
    int s = who ? __builtin_amdgcn_readlane(bi, (int)__builtin_ctzll(who)) : -1;
    if (who & (who - 1)) {  // equal candidates in several lanes: the first start
        uint32_t key = mine ? (uint32_t)bi : 0xffffffffu;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) key = min(key, (uint32_t)__shfl_xor((int)key, off, 64));
        s = (int)key;
    }
    if (lane == 0) {
        *dp_out = s >= 0 ? least : __builtin_inf();
        *bt_out = s >= 0 ? s + 1 : -1;
    }
}

__global__ __launch_bounds__(kDpThreads) void k_dp_level(int c, int K, int force, int bins, char* __restrict__ ws,
                                                         DpLayout L) {
    const int32_t* hdr = reinterpret_cast<const int32_t*>(ws);
    const size_t stride = (size_t)bins + 1;
    double* dp = reinterpret_cast<double*>(ws + L.dp);
    int32_t* bt = reinterpret_cast<int32_t*>(ws + L.bt);
    const DpArrays A{reinterpret_cast<const double*>(ws + L.pw), reinterpret_cast<const double*>(ws + L.pwx),
                     reinterpret_cast<const double*>(ws + L.pwx2), dp + (size_t)(c - 1) * stride};
    const int lane = threadIdx.x & 63;
    // ends 1 .. N; the last level needs only N.  Everything an end's first pass reads
    // is loaded before the header is looked at (the indices stay inside the arrays
    // for any end up to bins), so it is one trip to memory.
    const int e = c == K ? hdr[0] : (int)blockIdx.x * kDpWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + 1;
    const int lo = c - 1, top = c == 1 ? 0 : max(e - 1, lo);  // with one cluster, only start 1 has a predecessor
    double Pe = A.pw[e], PXe = A.pwx[e], PX2e = A.pwx2[e];
    DpPass d = dp_load(A, top, lo, lane);
    int N = hdr[0], status = hdr[1];
    double slack = *reinterpret_cast<const double*>(hdr + 2);
#pragma unroll
    for (int u = 0; u < kDpUnroll; ++u) __asm__ volatile("" : "+v"(d.p[u]), "+v"(d.px[u]), "+v"(d.px2[u]), "+v"(d.prev[u]));
    __asm__ volatile("" : "+v"(Pe), "+v"(PXe), "+v"(PX2e), "+v"(slack), "+v"(N), "+v"(status));
    N = __builtin_amdgcn_readfirstlane(N);
    if (__builtin_amdgcn_readfirstlane(status) != 0 || e > N) return;
    double* dp_out = dp + (size_t)c * stride + e;
    int32_t* bt_out = bt + (size_t)c * stride + e;
    if (e < c) {  // no segmentation of e points into c clusters
        if (lane == 0) {
            *dp_out = __builtin_inf();
            *bt_out = -1;
        }
        return;
    }
    if (force && c == 1) dp_end<-1>(d, Pe, PXe, PX2e, slack, top, lo, lane, A, dp_out, bt_out);
    else if (force && c == K) dp_end<1>(d, Pe, PXe, PX2e, slack, top, lo, lane, A, dp_out, bt_out);
    else dp_end<0>(d, Pe, PXe, PX2e, slack, top, lo, lane, A, dp_out, bt_out);
}

// jump[g][e]: where the backtrack stands after the kDpGroup levels K - 16 g ..
// K - 16 g - 15, starting them at end e; -1 where it breaks off.  Walking K levels
// one by one is K dependent loads (171 us for 256); the groups' walks run side by
// side, and k_dp_backtrack then takes 16 jumps and 16 short walks (8 + 11 us).
__global__ __launch_bounds__(256) void k_dp_jump(int K, int bins, char* __restrict__ ws, DpLayout L) {
    const int32_t* hdr = reinterpret_cast<const int32_t*>(ws);
    if (hdr[1] != 0) return;
    const int N = hdr[0];
    const size_t stride = (size_t)bins + 1;
    const int32_t* bt = reinterpret_cast<const int32_t*>(ws + L.bt);
    int32_t* jump = reinterpret_cast<int32_t*>(ws + L.jump);
    const int g = blockIdx.y, top = K - g * kDpGroup;
    // the first group starts at end N alone
    const int first = (int)blockIdx.x * 256 + (int)threadIdx.x;
    const int e0 = g == 0 ? (first == 0 ? N : N + 1) : first;
    if (e0 > N) return;
    int e = e0;
    for (int c = top; c > top - kDpGroup && c >= 1; --c) {
        const int s = e >= c ? bt[(size_t)c * stride + e] : -1;
        e = s - 1;
        if (s < 1) { e = -1; break; }
    }
    jump[(size_t)g * stride + e0] = e;
}

__global__ __launch_bounds__(kDpMaxK) void k_dp_backtrack(int K, int force, int bins, char* __restrict__ ws, DpLayout L,
                                                          float* __restrict__ out) {
    __shared__ int ends[kDpMaxK + 1];  // ends[c]: last point of cluster c; ends[0]: where cluster 1 begins
    __shared__ int start[kDpGroups];
    __shared__ int broken, unsorted;
    __shared__ float cbk[kDpMaxK];
    int32_t* hdr = reinterpret_cast<int32_t*>(ws);
    if (hdr[1] != 0) return;
    const int N = hdr[0], t = threadIdx.x;
    const size_t stride = (size_t)bins + 1;
    const double* pw = reinterpret_cast<const double*>(ws + L.pw);
    const double* pwx = reinterpret_cast<const double*>(ws + L.pwx);
    const int32_t* bt = reinterpret_cast<const int32_t*>(ws + L.bt);
    const int32_t* jump = reinterpret_cast<const int32_t*>(ws + L.jump);
    const int groups = (K + kDpGroup - 1) / kDpGroup;
    if (t == 0) {
        int e = N;
        broken = 0;
        for (int g = 0; g < groups; ++g) {
            start[g] = e;
            if (e < 0) broken = 1;
            else e = jump[(size_t)g * stride + e];
        }
        if (e < 0) broken = 1;
    }
    __syncthreads();
    if (broken) {
        if (t == 0) hdr[1] = 3;
        return;
    }
    if (t < groups) {
        int e = start[t];
        for (int c = K - t * kDpGroup; c > K - (t + 1) * kDpGroup && c >= 1; --c) {
            ends[c] = e;
            e = bt[(size_t)c * stride + e] - 1;
            if (c == 1) ends[0] = e;
        }
    }
    __syncthreads();
    if (t < K) {
        const int c = t + 1, e = ends[c], i = ends[c - 1];
        if (force && c == 1) cbk[t] = -1.0f;
        else if (force && c == K) cbk[t] = 1.0f;
        else cbk[t] = (float)((pwx[e] - pwx[i]) / (pw[e] - pw[i]));
    }
    __syncthreads();
    sort_codewords(cbk, K, out, &unsorted);
}

// ---------------------------------------------------------------------------
// Lloyd-Max accumulators (reference CUDA semantics; fp32 sums are order dependent).
// The block absmax skips NaN elements as the reference's running maximum does
// (lloyd_max_fused_kernel.cu:78-95, 141-158).
struct LloydLds {
    float thr[260];
    uint16_t bucket[4100];
};

// Codeword of a normalised value in the Lloyd kernels, as the reference's
// binary search picks it (lloyd_max_fused_kernel.cu:17-48): the lower bound k
// and its left neighbour k-1, ties to the left.  For x inside the codebook this
// is nearest_index.  It differs in two places: NaN (no codeword compares below
// it, and NaN distances fail the <= test) takes index 0, and x above the last
// codeword compares the last two entries instead of taking the last one.
__device__ __forceinline__ int lloyd_index(float x, const float* thr, const uint16_t* bucket, int K, float cb_prev,
                                           float cb_last) {
    if (x != x) return 0;
    if (K >= 2 && x > cb_last) return fabsf(x - cb_prev) <= fabsf(x - cb_last) ? K - 2 : K - 1;
    return nearest_index(x, thr, bucket, K);
}

template <typename G>
__global__ __launch_bounds__(256) void k_lloyd_accumulate(const G* __restrict__ g, int64_t nrows, int64_t period,
                                                          const CodebookTables* __restrict__ T,
                                                          float* __restrict__ sums,
                                                          unsigned long long* __restrict__ counts) {
    __shared__ LloydLds L;
    __shared__ float s_sum[256];
    __shared__ uint32_t s_cnt[256];
    const int K = T->K;
    const float cb_last = T->cb[K - 1], cb_prev = T->cb[K >= 2 ? K - 2 : 0];
    for (int i = threadIdx.x; i < 260; i += 256) L.thr[i] = T->thr[i];
    for (int i = threadIdx.x; i < 4100; i += 256) L.bucket[i] = T->bucket[i];
    s_sum[threadIdx.x] = 0.0f;
    s_cnt[threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < nrows; row += (int64_t)gridDim.x * 4) {
        const int64_t base = row * period;
        float amax = 0.0f;
        for (int64_t j = lane; j < period; j += 64) amax = max_skip_nan(amax, fabsf(to_f32(g[base + j])));
        amax = group_max_skip_nan(amax, 64);
        for (int64_t j = lane; j < period; j += 64) {
            const float v = to_f32(g[base + j]);
            const float x = (amax > 0.0f) ? v / amax : 0.0f;
            const int k = lloyd_index(x, L.thr, L.bucket, K, cb_prev, cb_last);
            atomicAdd(&s_sum[k], x);
            atomicAdd(&s_cnt[k], 1u);
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < K; k += 256) {
        if (s_cnt[k]) {
            atomicAdd(&sums[k], s_sum[k]);
            atomicAdd(&counts[k], (unsigned long long)s_cnt[k]);
        }
    }
}

template <typename G>
__global__ __launch_bounds__(256) void k_lloyd_mse(const G* __restrict__ g, int64_t nrows, int64_t period,
                                                   const CodebookTables* __restrict__ T,
                                                   const float* __restrict__ new_cb, float* __restrict__ mse_norm,
                                                   float* __restrict__ mse_orig) {
    __shared__ LloydLds L;
    __shared__ float red[2][4];
    const int K = T->K;
    const float cb_last = T->cb[K - 1], cb_prev = T->cb[K >= 2 ? K - 2 : 0];
    for (int i = threadIdx.x; i < 260; i += 256) L.thr[i] = T->thr[i];
    for (int i = threadIdx.x; i < 4100; i += 256) L.bucket[i] = T->bucket[i];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    float en = 0.0f, eo = 0.0f;
    for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < nrows; row += (int64_t)gridDim.x * 4) {
        const int64_t base = row * period;
        float amax = 0.0f;
        for (int64_t j = lane; j < period; j += 64) amax = max_skip_nan(amax, fabsf(to_f32(g[base + j])));
        amax = group_max_skip_nan(amax, 64);
        for (int64_t j = lane; j < period; j += 64) {
            const float v = to_f32(g[base + j]);
            const float x = (amax > 0.0f) ? v / amax : 0.0f;
            const int k = lloyd_index(x, L.thr, L.bucket, K, cb_prev, cb_last);
            const float err = x - new_cb[k];
            const float e2 = err * err;
            en = en + e2;
            const float oe = err * amax;
            const float o2 = oe * oe;
            eo = eo + o2;
        }
    }
    en = group_sum(en, 64);
    eo = group_sum(eo, 64);
    if (lane == 0) { red[0][threadIdx.x >> 6] = en; red[1][threadIdx.x >> 6] = eo; }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(mse_norm, (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]));
        atomicAdd(mse_orig, (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
    }
}

namespace {
int grid_for_rows(int64_t units, int cap) {
    int64_t g = (units + 3) / 4;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (int)g;
}
struct TempTables {
    void* ptr = nullptr;
    hipStream_t st = nullptr;
    int init(const float* cb, int K, hipStream_t s) {
        st = s;
        hipError_t e = device_malloc_async(&ptr, sizeof(CodebookTables), s);
        if (e != hipSuccess) return hip_status(e, "hipMallocAsync(codebook tables)");
        return gefen_prepare_codebook(cb, K, ptr, reinterpret_cast<gefen_stream_t>(s));
    }
    ~TempTables() {
        if (ptr) (void)hipFreeAsync(ptr, st);
    }
};

int check_rows(const void* g, int dt, int64_t numel, int64_t period) {
    if (!valid_dtype(dt)) return fail_inval("unsupported gradient dtype %d", dt);
    if (period <= 0) return fail_inval("Expected period to be positive, got %lld", (long long)period);
    if (numel < 0 || numel % period)
        return fail_inval("Expected grad_flat.numel()=%lld to be divisible by period=%lld", (long long)numel,
                          (long long)period);
    if (numel > 0 && !g) return fail_inval("null gradient pointer");
    return GEFEN_OK;
}
}  // namespace
}  // namespace gefen

using namespace gefen;

extern "C" size_t gefen_codebook_tables_size(void) { return sizeof(CodebookTables); }

extern "C" int gefen_prepare_codebook(const float* codebook, int codebook_size, void* tables,
                                      gefen_stream_t stream) {
    if (!codebook || !tables) return fail_inval("null pointer");
    if (codebook_size <= 0 || codebook_size > 256)
        return fail_inval("Expected codebook to have at most 256 entries, got %d", codebook_size);
    hipLaunchKernelGGL(k_prepare_codebook, dim3(1), dim3(kPrepThreads), 0, reinterpret_cast<hipStream_t>(stream), codebook,
                       codebook_size, static_cast<CodebookTables*>(tables));
    return launch_status("gefen_prepare_codebook");
}

namespace gefen {
namespace {
// The kernel of a row length: signs for rows of one element, W = 1 for rows shorter
// than a 16-byte vector, two vectors per lane up to half a wave's rows, eight up to
// 64 lanes of them, else rows read twice.
struct HistKind {
    int w, r, lpr_log2, nvec;  // r = -1: signs
};
HistKind hist_kind(int dtype, int64_t rowlen) {
    const int wide = dtype == GEFEN_F32 ? 4 : 8;
    if (rowlen == 1) return {wide, -1, 0, 0};
    const int w = rowlen < wide ? 1 : wide;
    const int64_t nvec = (rowlen + w - 1) / w;
    if (nvec > 64 * 8) return {1, 0, 6, 0};
    const int r = w == 1 || nvec > 64 * 2 ? 8 : 2;
    int l2 = 0;
    while ((int64_t)r << l2 < nvec) ++l2;
    return {w, r, l2, (int)nvec};
}

template <typename T, int WIDE>
hipError_t launch_histogram(const HistKind& k, const HistBatch& b, int grid, hipStream_t st) {
    if (k.r == -1) hipLaunchKernelGGL((k_histogram_signs<T, WIDE>), dim3(grid), dim3(256), 0, st, b);
    else if (k.r == 0) hipLaunchKernelGGL((k_histogram<T, 1, 0>), dim3(grid), dim3(256), 0, st, b);
    else if (k.w == 1) hipLaunchKernelGGL((k_histogram<T, 1, 8>), dim3(grid), dim3(256), 0, st, b);
    else if (k.r == 2) hipLaunchKernelGGL((k_histogram<T, WIDE, 2>), dim3(grid), dim3(256), 0, st, b);
    else hipLaunchKernelGGL((k_histogram<T, WIDE, 8>), dim3(grid), dim3(256), 0, st, b);
    return hipGetLastError();
}

// Task i adds to counts + i * stride.
int run_histograms(const gefen_histogram_task* tasks, int ntasks, int64_t* counts, int64_t stride, int bins,
                   hipStream_t st) {
    for (int i = 0; i < ntasks; ++i) {
        const int rc = check_rows(tasks[i].grad, tasks[i].dtype, tasks[i].numel, tasks[i].period);
        if (rc) return rc;
    }
    std::vector<char> done(ntasks, 0);
    for (int i = 0; i < ntasks; ++i) {
        if (done[i] || tasks[i].numel == 0) continue;
        const HistKind kind = hist_kind(tasks[i].dtype, tasks[i].period);
        HistBatch b;
        memset(&b, 0, sizeof(b));
        b.bins = bins;
        b.bw = (float)(2.0 / (double)bins);
        b.pow2 = (bins & (bins - 1)) == 0;
        b.scale = (float)bins * 0.5f;
        int64_t wg = 0;
        for (int j = i; j < ntasks && b.ntasks < kHistTasks; ++j) {
            const gefen_histogram_task& t = tasks[j];
            if (done[j] || t.numel == 0 || t.dtype != tasks[i].dtype) continue;
            const HistKind k = hist_kind(t.dtype, t.period);
            if (k.w != kind.w || k.r != kind.r) continue;
            HistTask& o = b.t[b.ntasks];
            o.g = t.grad;
            o.counts = reinterpret_cast<unsigned long long*>(counts + (int64_t)j * stride);
            o.nrows = t.numel / t.period;
            o.rowlen = t.period;
            o.nvec = k.nvec;
            o.lpr_log2 = k.lpr_log2;
            b.wg_begin[b.ntasks++] = (int32_t)wg;
            // every workgroup adds its counts to the tensor's at the end: no more of them
            // than fill the chip, each with 16384 elements or more (signs: three sums)
            wg += std::max<int64_t>(1, std::min<int64_t>(kHistMaxWgs, t.numel / 16384));
            done[j] = 1;
        }
        b.wg_begin[b.ntasks] = (int32_t)wg;
        hipError_t e;
        if (tasks[i].dtype == GEFEN_F32) e = launch_histogram<float, 4>(kind, b, (int)wg, st);
        else if (tasks[i].dtype == GEFEN_BF16) e = launch_histogram<bf16_t, 8>(kind, b, (int)wg, st);
        else e = launch_histogram<f16_t, 8>(kind, b, (int)wg, st);
        if (e != hipSuccess) return hip_status(e, "gefen_exact_histogram");
    }
    return GEFEN_OK;
}
}  // namespace
}  // namespace gefen

extern "C" int gefen_exact_histogram(const void* grad, int grad_dtype, int64_t numel, int64_t period,
                                     int64_t* bin_counts, int bins, gefen_stream_t stream) {
    int rc = check_rows(grad, grad_dtype, numel, period);
    if (rc) return rc;
    if (bins <= 0 || bins > kHistBins) return fail_inval("Expected histogram bins in [1, 4096], got %d", bins);
    if (!bin_counts) return fail_inval("null bin_counts");
    gefen_histogram_task t;
    memset(&t, 0, sizeof(t));
    t.grad = grad;
    t.numel = numel;
    t.period = period;
    t.dtype = grad_dtype;
    return run_histograms(&t, 1, bin_counts, 0, bins, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int gefen_exact_histogram_tasks(const gefen_histogram_task* tasks, int ntasks, float* acc, int bins,
                                           int64_t* counts, gefen_stream_t stream) {
    if (ntasks < 0 || (ntasks > 0 && !tasks)) return fail_inval("invalid task array");
    if (bins <= 0 || bins > kHistBins) return fail_inval("Expected histogram bins in [1, 4096], got %d", bins);
    if (ntasks == 0) return GEFEN_OK;
    if (!acc || !counts) return fail_inval("null pointer");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int64_t n = (int64_t)ntasks * bins;
    hipLaunchKernelGGL(k_zero_i64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, counts, n);
    int rc = launch_status("gefen_exact_histogram_tasks (zero)");
    if (rc) return rc;
    rc = run_histograms(tasks, ntasks, counts, bins, bins, st);
    if (rc) return rc;
    hipLaunchKernelGGL(k_accumulate_tasks, dim3((bins + 63) / 64), dim3(64), 0, st, acc, counts, ntasks, bins);
    return launch_status("gefen_exact_histogram_tasks (sum)");
}

extern "C" int gefen_accumulate_counts(float* acc, const int64_t* counts, int bins, gefen_stream_t stream) {
    if (!acc || !counts || bins <= 0) return fail_inval("invalid histogram accumulation arguments");
    hipLaunchKernelGGL(k_accumulate_counts, dim3((bins + 255) / 256), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), acc, counts, bins);
    return launch_status("gefen_accumulate_counts");
}

extern "C" size_t gefen_exact_dp_workspace_size(int bins, int codebook_size) {
    if (bins <= 0 || codebook_size <= 0) return 0;
    return DpLayout(bins, codebook_size).total;
}

extern "C" int gefen_exact_dp(const float* counts, int bins, int codebook_size, int force_endpoints,
                              float* codebook_out, void* workspace, gefen_stream_t stream) {
    if (!counts || !codebook_out || !workspace) return fail_inval("null pointer");
    if (bins <= 0 || bins > 4096 || (bins & (bins - 1)))
        return fail_inval("exact DP needs a power-of-two bin count <= 4096, got %d", bins);
    if (codebook_size <= 0 || codebook_size > 256)
        return fail_inval("Expected codebook to have at most 256 entries, got %d", codebook_size);
    const int K = codebook_size;
    DpLayout L(bins, K);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    hipLaunchKernelGGL(k_dp_init, dim3(1), dim3(kDpInitThreads), 0, st, counts, bins, K, force_endpoints ? 1 : 0,
                       ws, L, codebook_out);
    int rc = launch_status("gefen_exact_dp init");
    if (rc) return rc;
    // one wave per end (at most bins ends); the last level has one end
    const int grid = (bins + kDpWaves - 1) / kDpWaves;
    for (int c = 1; c <= K; ++c) {
        hipLaunchKernelGGL(k_dp_level, dim3(c == K ? 1 : grid), dim3(c == K ? 64 : kDpThreads), 0, st, c, K,
                           force_endpoints ? 1 : 0, bins, ws, L);
        rc = launch_status("gefen_exact_dp level");
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_dp_jump, dim3(bins / 256 + 1, (K + kDpGroup - 1) / kDpGroup), dim3(256), 0, st, K, bins, ws, L);
    rc = launch_status("gefen_exact_dp jump");
    if (rc) return rc;
    hipLaunchKernelGGL(k_dp_backtrack, dim3(1), dim3(kDpMaxK), 0, st, K, force_endpoints ? 1 : 0, bins, ws, L,
                       codebook_out);
    return launch_status("gefen_exact_dp backtrack");
}

extern "C" int gefen_lloyd_accumulate(const void* grad, int grad_dtype, int64_t numel, int64_t period,
                                      const float* codebook, int codebook_size, float* sums, int64_t* counts,
                                      gefen_stream_t stream) {
    int rc = check_rows(grad, grad_dtype, numel, period);
    if (rc) return rc;
    if (!codebook || !sums || !counts) return fail_inval("null pointer");
    if (codebook_size <= 0 || codebook_size > 256)
        return fail_inval("Expected codebook to have at most 256 entries, got %d", codebook_size);
    if (numel == 0) return GEFEN_OK;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    TempTables tt;
    rc = tt.init(codebook, codebook_size, st);
    if (rc) return rc;
    const int64_t nrows = numel / period;
    const int grid = grid_for_rows(nrows, 2048);
    auto* T = static_cast<const CodebookTables*>(tt.ptr);
    auto* cnt = reinterpret_cast<unsigned long long*>(counts);
    if (grad_dtype == GEFEN_F32)
        hipLaunchKernelGGL(k_lloyd_accumulate<float>, dim3(grid), dim3(256), 0, st, static_cast<const float*>(grad),
                           nrows, period, T, sums, cnt);
    else if (grad_dtype == GEFEN_BF16)
        hipLaunchKernelGGL(k_lloyd_accumulate<bf16_t>, dim3(grid), dim3(256), 0, st,
                           static_cast<const bf16_t*>(grad), nrows, period, T, sums, cnt);
    else
        hipLaunchKernelGGL(k_lloyd_accumulate<f16_t>, dim3(grid), dim3(256), 0, st, static_cast<const f16_t*>(grad),
                           nrows, period, T, sums, cnt);
    return launch_status("gefen_lloyd_accumulate");
}

extern "C" int gefen_lloyd_mse(const void* grad, int grad_dtype, int64_t numel, int64_t period,
                               const float* old_codebook, const float* new_codebook, int codebook_size,
                               float* mse_normalized_sum, float* mse_original_sum, gefen_stream_t stream) {
    int rc = check_rows(grad, grad_dtype, numel, period);
    if (rc) return rc;
    if (!old_codebook || !new_codebook || !mse_normalized_sum || !mse_original_sum) return fail_inval("null pointer");
    if (codebook_size <= 0 || codebook_size > 256)
        return fail_inval("Expected codebook to have at most 256 entries, got %d", codebook_size);
    if (numel == 0) return GEFEN_OK;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    TempTables tt;
    rc = tt.init(old_codebook, codebook_size, st);
    if (rc) return rc;
    const int64_t nrows = numel / period;
    const int grid = grid_for_rows(nrows, 2048);
    auto* T = static_cast<const CodebookTables*>(tt.ptr);
    if (grad_dtype == GEFEN_F32)
        hipLaunchKernelGGL(k_lloyd_mse<float>, dim3(grid), dim3(256), 0, st, static_cast<const float*>(grad), nrows,
                           period, T, new_codebook, mse_normalized_sum, mse_original_sum);
    else if (grad_dtype == GEFEN_BF16)
        hipLaunchKernelGGL(k_lloyd_mse<bf16_t>, dim3(grid), dim3(256), 0, st, static_cast<const bf16_t*>(grad), nrows,
                           period, T, new_codebook, mse_normalized_sum, mse_original_sum);
    else
        hipLaunchKernelGGL(k_lloyd_mse<f16_t>, dim3(grid), dim3(256), 0, st, static_cast<const f16_t*>(grad), nrows,
                           period, T, new_codebook, mse_normalized_sum, mse_original_sum);
    return launch_status("gefen_lloyd_mse");
}
