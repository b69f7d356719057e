// Partition-block statistics for the automatic period (partitioning.py).
//
// Score of a divisor p of n (partitioning.py:43-78): with L_i = log(x_i + eps),
// m_j the mean of L over block j of p elements, score = mean_j |m_{j+1} - m_j|.
// The logarithms and everything that is large happen in one pass over the
// values (k_score_pass): a workgroup holds the logarithms of a chunk of Q elements
// in LDS and forms the block sums and adjacent differences of the small divisors
// (up to kPassMax) there, each from its largest listed divisor.  Small divisors that
// do not fit take another pass.  The others come from block sums that a pass stored
// (k_score_derived), in two stages, and those that share too little with a pass from
// the values (k_log_block_sums).  k_score_final adds the parts up.  float64 throughout, in
// a fixed order, with no host synchronisation; the scores agree with numpy's
// pairwise sums to ~1e-15 relative.
// (One launch and one pass over stored sums per divisor, from the logarithms of all
// elements written out, took 16 B of workspace per element and about 60 B of
// traffic: all 25 divisors of 64M float32 values 1.18 ms, now 0.27, and GPT-2 124M's
// 111 gradients 4400 launches, now 40.)
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "capi_internal.h"
#include "common.h"

namespace gefen {

// x of one element: mode 0 = f64(f32(v)); 1 = f64(f32(v)*f32(v)); 2 = f64(f32(v))^2
template <typename T>
__device__ __forceinline__ double transform(T raw, int mode) {
    const float v = to_f32(raw);
    if (mode == 1) {
        const float sq = v * v;
        return (double)sq;
    }
    const double d = (double)v;
    if (mode == 2) return d * d;
    return d;
}

// Natural logarithm of a positive, finite, normal y by an accurate table (S. Gal,
// "Computing elementary functions", 1986), arranged as the log of Arm's Optimized
// Routines is (an interval's index from the bits below an offset that is subtracted, a
// two-part ln 2); the entries are this file's own and the polynomial is the plain
// series.  y = z 2^e with z in [0.6875, 1.375), c
// the table's reciprocal of z's interval, log y = (e ln 2 - log c) + log1p(z c - 1).
// The entries are chosen so that -log c is a multiple of 2^-42 to within 2^-64, and
// ln 2 is split at the same bit, so the bracket is exact; the intervals beside 1
// have c = 1, which keeps the relative error there.  Below 1 ulp everywhere,
// 0.250 ulp on average (3e7 values; glibc's log: 0.250).  22 instructions where the
// library's log takes 108, which bound the scores: 64M float32 values' base sums 271 us.
struct LogEntry { double c, l; };
__device__ const LogEntry kLogTable[128] = {
    {0x1.734f0c50379d1p+0, -0x1.7cc7f7d080000p-2}, {0x1.713786d4afec1p+0, -0x1.76feecab27000p-2},
    {0x1.6f26016aa87b7p+0, -0x1.713e3397e4000p-2}, {0x1.6d1a6265104ffp+0, -0x1.6b85b4c76e000p-2},
    {0x1.6b1490a738057p+0, -0x1.65d558cc6a000p-2}, {0x1.691473a474524p+0, -0x1.602d08a36b000p-2},
    {0x1.6719f35b5c3d0p+0, -0x1.5a8cadae73000p-2}, {0x1.6524f84f148aap+0, -0x1.54f431aa7b000p-2},
    {0x1.63356b832e4ecp+0, -0x1.4f637eabd5000p-2}, {0x1.614b367f75e7ep+0, -0x1.49da7f313c000p-2},
    {0x1.5f66433e1024ep+0, -0x1.44591df815000p-2}, {0x1.5d867c3b3d9b0p+0, -0x1.3edf4631a5000p-2},
    {0x1.5babcc60579c7p+0, -0x1.396ce34d7e000p-2}, {0x1.59d61f0b811b0p+0, -0x1.3401e116fd000p-2},
    {0x1.58056010e4100p+0, -0x1.2e9e2bc059000p-2}, {0x1.56397ba1016e6p+0, -0x1.2941af9d49000p-2},
    {0x1.54725e6551e7ep+0, -0x1.23ec597eac000p-2}, {0x1.52aff564c9e1dp+0, -0x1.1e9e166744000p-2},
    {0x1.50f22e0d557ddp+0, -0x1.1956d3ae42000p-2}, {0x1.4f38f628b6d80p+0, -0x1.14167ee3c6000p-2},
    {0x1.4d843be8f5e4ap+0, -0x1.0edd05fcbb000p-2}, {0x1.4bd3edd802744p+0, -0x1.09aa572704000p-2},
    {0x1.4a27fad6105e5p+0, -0x1.047e60c9d7000p-2}, {0x1.4880521c549d1p+0, -0x1.feb2232740000p-3},
    {0x1.46dce3415f42ap+0, -0x1.f474b11a78000p-3}, {0x1.453d9e282746ap+0, -0x1.ea4449d522000p-3},
    {0x1.43a2730a8bbf0p+0, -0x1.e020cc60f2000p-3}, {0x1.420b525ed9bd2p+0, -0x1.d60a17cc34000p-3},
    {0x1.40782d0e57fa3p+0, -0x1.cc000c8d5e000p-3}, {0x1.3ee8f42945333p+0, -0x1.c2028aaa88000p-3},
    {0x1.3d5d991520816p+0, -0x1.b81172e7d8000p-3}, {0x1.3bd60d8e2e75ap+0, -0x1.ae2ca6dc68000p-3},
    {0x1.3a52438784311p+0, -0x1.a454082d64000p-3}, {0x1.38d22d33bdeabp+0, -0x1.9a8778cd7a000p-3},
    {0x1.3755bd16f121dp+0, -0x1.90c6db7ab6000p-3}, {0x1.35dce5f42827cp+0, -0x1.8712134ec8000p-3},
    {0x1.34679ac8800c8p+0, -0x1.7d6903a668000p-3}, {0x1.32f5ced247c82p+0, -0x1.73cb9057f4000p-3},
    {0x1.3187758b806a3p+0, -0x1.6a399d96d6000p-3}, {0x1.301c82aa9efe5p+0, -0x1.60b3100010000p-3},
    {0x1.2eb4ea19559bdp+0, -0x1.5737cc6380000p-3}, {0x1.2d50a00ea687ep+0, -0x1.4dc7b87b50000p-3},
    {0x1.2bef98e143c5cp+0, -0x1.4462b9bebe000p-3}, {0x1.2a91c92ad0032p+0, -0x1.3b08b6572a000p-3},
    {0x1.293725b7508c7p+0, -0x1.31b994b6cc000p-3}, {0x1.27dfa383e0b08p+0, -0x1.28753b95f2000p-3},
    {0x1.268b37c9ec2d7p+0, -0x1.1f3b924724000p-3}, {0x1.2539d7e750aedp+0, -0x1.160c80184a000p-3},
    {0x1.23eb796eb5497p+0, -0x1.0ce7ecc97c000p-3}, {0x1.22a01226530cfp+0, -0x1.03cdc08b30000p-3},
    {0x1.2157980196dc9p+0, -0x1.f57bc7af80000p-4}, {0x1.2012011dc0aa8p+0, -0x1.e3707ec210000p-4},
    {0x1.1ecf43c4b44aap+0, -0x1.d179785348000p-4}, {0x1.1d8f566f1dcb8p+0, -0x1.bf968733d0000p-4},
    {0x1.1c522fbdd7d53p+0, -0x1.adc77eac9c000p-4}, {0x1.1b17c67ac34b7p+0, -0x1.9c0c32950c000p-4},
    {0x1.19e0119c95e68p+0, -0x1.8a64779480000p-4}, {0x1.18ab08367b541p+0, -0x1.78d0223ef0000p-4},
    {0x1.1778a1900f719p+0, -0x1.674f087ac8000p-4}, {0x1.1648d50bc916dp+0, -0x1.55e1001658000p-4},
    {0x1.151b9a39e7c81p+0, -0x1.4485dfe5a8000p-4}, {0x1.13f0e8ce5b9fcp+0, -0x1.333d7f38a4000p-4},
    {0x1.12c8b89b7821bp+0, -0x1.2207b594fc000p-4}, {0x1.11a301966afd2p+0, -0x1.10e45b0040000p-4},
    {0x1.107fbbda4c119p+0, -0x1.ffa6906d48000p-5}, {0x1.0f5edfa926769p+0, -0x1.dda8ad88b8000p-5},
    {0x1.0e40655273e26p+0, -0x1.bbcebf19e8000p-5}, {0x1.0d2445617a8cap+0, -0x1.9a187b1e40000p-5},
    {0x1.0c0a78636df4ap+0, -0x1.7885950228000p-5}, {0x1.0af2f720c1cb6p+0, -0x1.5715c47d78000p-5},
    {0x1.09ddba6797875p+0, -0x1.35c8bf4200000p-5}, {0x1.08cabb33f25eep+0, -0x1.149e3dd720000p-5},
    {0x1.07b9f2978ced6p+0, -0x1.e72bf18850000p-6}, {0x1.06ab59c1ca313p+0, -0x1.a55f532400000p-6},
    {0x1.059eea0381c6dp+0, -0x1.63d616a230000p-6}, {0x1.04949cbfc56cep+0, -0x1.228fb19840000p-6},
    {0x1.038c6b7522cdfp+0, -0x1.c31736d0e0000p-7}, {0x1.02864fc596b26p+0, -0x1.41929eaae0000p-7},
    {0x1.0182435f388e2p+0, -0x1.81211b6f40000p-8}, {0x1.0000000000000p+0, 0x0.0p+0},
    {0x1.0000000000000p+0, 0x0.0p+0}, {0x1.fa11ca965839fp-1, 0x1.7dc4787140000p-7},
    {0x1.f6310ac059155p-1, 0x1.3cea457110000p-6}, {0x1.f25f643f59d40p-1, 0x1.b9fc02d850000p-6},
    {0x1.ee9c7f79f1d8ep-1, 0x1.1b0d993e88000p-5}, {0x1.eae807a334a1ep-1, 0x1.58a5bb8910000p-5},
    {0x1.e741aa5665b98p-1, 0x1.95c8312000000p-5}, {0x1.e3a91796954bep-1, 0x1.d276b92730000p-5},
    {0x1.e01e01e000bc6p-1, 0x1.0759835a88000p-4}, {0x1.dca01dc30ada0p-1, 0x1.253f632c7c000p-4},
    {0x1.d92f222cb17e8p-1, 0x1.42edcc1784000p-4}, {0x1.d5cac80117fa1p-1, 0x1.60658ac9ec000p-4},
    {0x1.d272ca3af5339p-1, 0x1.7da76701f8000p-4}, {0x1.cf26e5bf09694p-1, 0x1.9ab4249088000p-4},
    {0x1.cbe6d95fc33d5p-1, 0x1.b78c82be2c000p-4}, {0x1.c8b265ac4c2d4p-1, 0x1.d4313d8580000p-4},
    {0x1.c5894d0a5e22dp-1, 0x1.f0a30c3b74000p-4}, {0x1.c26b538e50679p-1, 0x1.0671514190000p-3},
    {0x1.bf583edef19ecp-1, 0x1.14785871ca000p-3}, {0x1.bc4fd64f720b7p-1, 0x1.2266f1ba74000p-3},
    {0x1.b951e2a9951d9p-1, 0x1.303d71b350000p-3}, {0x1.b65e2e38127d9p-1, 0x1.3dfc2b20d6000p-3},
    {0x1.b37484a8acf13p-1, 0x1.4ba36f5058000p-3}, {0x1.b094b31a8b69bp-1, 0x1.59338da7d6000p-3},
    {0x1.adbe87f5bc9b8p-1, 0x1.66acd43814000p-3}, {0x1.aaf1d2f3a7801p-1, 0x1.740f8f6b3c000p-3},
    {0x1.a82e650b4d5bbp-1, 0x1.815c0a39a4000p-3}, {0x1.a574106e9f734p-1, 0x1.8e928e0ef8000p-3},
    {0x1.a2c2a87792586p-1, 0x1.9bb362ff18000p-3}, {0x1.a01a019cf1f83p-1, 0x1.a8becfd80c000p-3},
    {0x1.9d79f172be74cp-1, 0x1.b5b519fca4000p-3}, {0x1.9ae24ea218c97p-1, 0x1.c2968568ce000p-3},
    {0x1.9852f0d364f53p-1, 0x1.cf6354fc56000p-3}, {0x1.95cbb0b883533p-1, 0x1.dc1bca2788000p-3},
    {0x1.934c67f45a83fp-1, 0x1.e8c02545ca000p-3}, {0x1.90d4f11ce552ep-1, 0x1.f550a57514000p-3},
    {0x1.8e6527a98ff44p-1, 0x1.00e6c46901000p-2}, {0x1.8bfce8021894dp-1, 0x1.071b86076a000p-2},
    {0x1.899c0f5ac9355p-1, 0x1.0d46b5877c000p-2}, {0x1.87427bc7638d0p-1, 0x1.1368703564000p-2},
    {0x1.84f00c2075725p-1, 0x1.1980d2efcd000p-2}, {0x1.82a4a01169098p-1, 0x1.1f8ff9f66e000p-2},
    {0x1.806017feafd15p-1, 0x1.2596012177000p-2}, {0x1.7e225513283c9p-1, 0x1.2b9303b234000p-2},
    {0x1.7beb391e398aep-1, 0x1.31871ca1cd000p-2}, {0x1.79baa6b60d78ep-1, 0x1.3772663a75000p-2},
    {0x1.779081163d694p-1, 0x1.3d54fa657c000p-2}, {0x1.756cac1dbdd05p-1, 0x1.432ef2a6c0000p-2}
};

__device__ __forceinline__ bool table_log_takes(double y) {  // not zero, negative, subnormal, inf or NaN
    return (uint32_t)(__builtin_bit_cast(uint64_t, y) >> 32) - 0x00100000u < 0x7fe00000u;
}
__device__ __forceinline__ double table_log(double y, const LogEntry* table) {
    const uint64_t b = __builtin_bit_cast(uint64_t, y);
    const uint64_t t = b - 0x3fe6000000000000ull;
    const LogEntry E = table[(t >> 45) & 127];
    const double z = __builtin_bit_cast(double, b - (t & 0xfff0000000000000ull));
    const double e = (double)((int32_t)(t >> 32) >> 20);
    const double r = __builtin_fma(z, E.c, -1.0);
    const double hi = __builtin_fma(e, 0x1.62e42fefa3800p-1, E.l);
    double q = __builtin_fma(r, -0.125, 1.0 / 7.0);
    q = __builtin_fma(r, q, -1.0 / 6.0);
    q = __builtin_fma(r, q, 0.2);
    q = __builtin_fma(r, q, -0.25);
    q = __builtin_fma(r, q, 1.0 / 3.0);
    q = __builtin_fma(r, q, -0.5);
    return hi + __builtin_fma(r * r, q, __builtin_fma(e, 0x1.ef35793c76730p-45, r));
}

constexpr int kScoreThreads = 256;
constexpr int kScoreBudget = 4096;  // float64 sums a chunk keeps in LDS (32 KB: four workgroups per CU)
constexpr int kScoreChunk = 2048;   // elements of a chunk, at most
constexpr int kScoreItems = 14;     // divisors of one pass (an accumulator and five scalars each)
// Largest divisor that a pass forms itself: the next ones have too few blocks in a
// chunk for a workgroup, and cost less from stored sums (all 25 divisors of 64M
// float32 values: 411 us with every divisor of the chunk in the pass).
constexpr int kPassMax = 48;
constexpr int kScorePer = 8;        // elements of a chunk per thread, at most
constexpr int kScoreTensors = 128;  // tensors of one launch (their addresses travel in the kernel arguments)

// One pass: chunks of Q consecutive elements (the last one shorter, a multiple of
// every item's p too); item 0 is the element level.
struct ScoreItem {
    int32_t count;   // blocks per chunk: Q / p
    int32_t tail;    // blocks of the last chunk
    int32_t parent;  // LDS offset of the item it is summed from
    int32_t ratio;   // p / parent's p
    int32_t at;      // LDS offset of its sums
    int64_t store;   // workspace offset (doubles) of its sums over the whole tensor, or -1
    int32_t rec;     // its record among the pass's scored items, or -1
    int32_t level;   // items of one level depend on lower levels only
    int32_t pad;
};
struct ScorePass {
    const void* values[kScoreTensors];
    double* ws;          // tensor t's workspace is ws + t * stride
    int64_t stride;
    int64_t nchunks;
    int64_t rec_off;     // records: 3 arrays of nunits (sum of differences, first sum, last sum) per scored item
    int64_t bad_off;     // per unit: elements with x + eps <= 0; -1 if another pass counts them
    double eps;
    int32_t q, tail;     // elements of a chunk, of the last one
    int32_t nitems, chunks_per_unit, nunits, pad;
    ScoreItem item[kScoreItems];
};
static_assert(sizeof(ScorePass) <= 4000, "kernel arguments are limited to 4 KB");

// A unit of consecutive chunks per workgroup, carried over from chunk to chunk; the
// differences between units are formed from the records.  Bound by instructions:
// about 30 vector instructions per element for the logarithm and its input, and 40
// for the sums and differences of six to fourteen divisors; the next chunk's loads
// run meanwhile (without them 12% slower).  64M float32 values: 230 us.
template <typename T, int MODE>
__global__ __launch_bounds__(kScoreThreads, 4) void k_score_pass(const ScorePass P) {
    __shared__ __attribute__((aligned(16))) double S[kScoreBudget];
    __shared__ __attribute__((aligned(16))) LogEntry table[128];
    __shared__ ScoreItem items[kScoreItems];  // from LDS: kept in scalar registers they spill
    __shared__ double last[kScoreItems];
    __shared__ double red[kScoreItems + 1][kScoreThreads / 64];
    const int t = threadIdx.x;
    if (t < 128) table[t] = kLogTable[t];
    if (t < P.nitems) items[t] = P.item[t];
    const T* __restrict__ src = static_cast<const T*>(P.values[blockIdx.y]);
    double* __restrict__ ws = P.ws + blockIdx.y * P.stride;
    const int64_t c0 = (int64_t)blockIdx.x * P.chunks_per_unit;
    const int64_t c1 = min(c0 + P.chunks_per_unit, P.nchunks);
    double acc[kScoreItems];
#pragma unroll
    for (int k = 0; k < kScoreItems; ++k) acc[k] = 0.0;
    double bad = 0.0;
    // the next chunk's elements are loaded while this one's sums are formed
    T raw[kScorePer];
    auto load = [&](int64_t c) {
        const int len = c + 1 == P.nchunks ? P.tail : P.q;
        const T* __restrict__ v = src + c * P.q;
#pragma unroll
        for (int u = 0; u < kScorePer; ++u) raw[u] = v[min(t + kScoreThreads * u, len - 1)];
    };
    load(c0);
    __syncthreads();
    for (int64_t c = c0; c < c1; ++c) {
        const bool tail = c + 1 == P.nchunks;
        const int len = tail ? P.tail : P.q;
#pragma unroll
        for (int u = 0; u < kScorePer; ++u) {
            if (t + kScoreThreads * u < len) {
                const double y = transform(raw[u], MODE) + P.eps;
                double l = table_log(y, table);
                if (!table_log_takes(y)) {
                    if (y <= 0.0) bad = bad + 1.0;  // numpy / the reference: NaN does not count
                    l = log(y);
                }
                S[t + kScoreThreads * u] = l;
            }
        }
        if (c + 1 < c1) load(c + 1);
        int level = 0;
        for (int k = 1; k < P.nitems; ++k) {
            const ScoreItem I = items[k];
            if (I.level != level) {
                __syncthreads();
                level = I.level;
            }
            const int cnt = tail ? I.tail : I.count;
            if (I.ratio == 2) {
                for (int j = t; j < cnt; j += kScoreThreads)
                    S[I.at + j] = S[I.parent + 2 * j] + S[I.parent + 2 * j + 1];
            } else {
                for (int j = t; j < cnt; j += kScoreThreads) {
                    const double* x = S + I.parent + j * I.ratio;
                    double s = x[0];
                    for (int u = 1; u < I.ratio; ++u) s = s + x[u];
                    S[I.at + j] = s;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kScoreItems; ++k) {
            if (k < P.nitems) {
                const ScoreItem I = items[k];
                const double* x = S + I.at;
                const int cnt = tail ? I.tail : I.count;
                if (I.store >= 0)
                    for (int j = t; j < cnt; j += kScoreThreads) ws[I.store + c * I.count + j] = x[j];
                if (I.rec >= 0) {
                    for (int j = t; j < cnt - 1; j += kScoreThreads) acc[k] = acc[k] + fabs(x[j + 1] - x[j]);
                    if (t == k) {
                        if (c > c0) acc[k] = acc[k] + fabs(x[0] - last[k]);
                        else ws[P.rec_off + (3 * (int64_t)I.rec + 1) * P.nunits + blockIdx.x] = x[0];
                        last[k] = x[cnt - 1];
                    }
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < kScoreItems; ++k) {
        if (k < P.nitems && items[k].rec >= 0) {
            double s = acc[k];
            for (int off = 32; off > 0; off >>= 1) s = s + __shfl_xor(s, off, 64);
            if ((t & 63) == 0) red[k][t >> 6] = s;
        }
    }
    for (int off = 32; off > 0; off >>= 1) bad = bad + __shfl_xor(bad, off, 64);
    if ((t & 63) == 0) red[kScoreItems][t >> 6] = bad;
    __syncthreads();
    if (t < P.nitems && items[t].rec >= 0) {
        double* rec = ws + P.rec_off + 3 * (int64_t)items[t].rec * P.nunits + blockIdx.x;
        rec[0] = (red[t][0] + red[t][1]) + (red[t][2] + red[t][3]);
        rec[2 * (int64_t)P.nunits] = last[t];
    }
    if (t == kScoreItems && P.bad_off >= 0)
        ws[P.bad_off + blockIdx.x] = (red[t][0] + red[t][1]) + (red[t][2] + red[t][3]);
}
static_assert(kScoreThreads == 256 && kScoreThreads * kScorePer == kScoreChunk, "four waves, a chunk in registers");

// out[j] = sum of log(x + eps) over block j of p elements, from the values: for
// divisors that share too little with a pass (multiples of a prime above kPassMax).
// A wave per block; each lane sums its strided items in order, then a butterfly.
// `bad`: where blocks count x + eps <= 0, or null.
template <typename T>
__global__ __launch_bounds__(256) void k_log_block_sums(const T* __restrict__ src, int64_t nblocks, int64_t p, int mode,
                                                        double eps, double* __restrict__ out, double* __restrict__ bad) {
    __shared__ __attribute__((aligned(16))) LogEntry table[128];
    if (threadIdx.x < 128) table[threadIdx.x] = kLogTable[threadIdx.x];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); blk < nblocks; blk += (int64_t)gridDim.x * 4) {
        const T* __restrict__ v = src + blk * p;
        double s = 0.0, b = 0.0;
        for (int64_t j = lane; j < p; j += 64) {
            const double y = transform(v[j], mode) + eps;
            if (y <= 0.0) b = b + 1.0;
            s = s + (table_log_takes(y) ? table_log(y, table) : log(y));
        }
        for (int off = 32; off > 0; off >>= 1) s = s + __shfl_xor(s, off, 64);
        if (lane == 0) out[blk] = s;
        if (bad) {
            for (int off = 32; off > 0; off >>= 1) b = b + __shfl_xor(b, off, 64);
            if (lane == 0) bad[blk] = b;
        }
    }
}

// Divisors summed from stored block sums: blocks of `ratio` entries of src, and the
// sum of |S[j+1] - S[j]| of each workgroup's share of the differences.
constexpr int kDerivedMax = 56;
constexpr int kDerivedTile = 1024;  // block sums in LDS at a time
struct DerivedItem {
    int64_t src;    // workspace offset of the source's sums
    int64_t ratio;  // source entries per block
    int64_t nblocks;
    int64_t part;   // workspace offset of this divisor's partial sums, one per workgroup
    int64_t store;  // workspace offset of its block sums for a later stage, or -1
};
struct DerivedBatch {
    double* ws;
    int64_t stride;
    int32_t count, pad;
    DerivedItem item[kDerivedMax];
    int32_t wg_begin[kDerivedMax + 1];
};
static_assert(sizeof(DerivedBatch) <= 4000, "kernel arguments are limited to 4 KB");

__global__ __launch_bounds__(256) void k_score_derived(const DerivedBatch B) {
    __shared__ double sums[kDerivedTile + 1];
    __shared__ double red[4];
    int lo_t = 0, hi_t = B.count - 1;
    while (lo_t < hi_t) {
        const int mid = (lo_t + hi_t + 1) >> 1;
        if (B.wg_begin[mid] <= (int)blockIdx.x) lo_t = mid;
        else hi_t = mid - 1;
    }
    const DerivedItem I = B.item[lo_t];
    double* ws = B.ws + blockIdx.y * B.stride;
    const double* __restrict__ src = ws + I.src;
    const int nwg = B.wg_begin[lo_t + 1] - B.wg_begin[lo_t], wb = (int)blockIdx.x - B.wg_begin[lo_t];
    const int64_t ndiff = I.nblocks - 1, per = (ndiff + nwg - 1) / nwg;
    const int64_t d0 = (int64_t)wb * per, d1 = min(d0 + per, ndiff);
    int l2 = 0;  // lanes per block: a power of two up to the wave
    while ((1LL << l2) < I.ratio && l2 < 6) ++l2;
    const int lane = threadIdx.x & 63, lpr = 1 << l2, rpw = 64 >> l2;
    double s = 0.0;
    for (int64_t d = d0; d < d1; d += kDerivedTile) {
        // differences d .. d + m - 1 need block sums d .. d + m
        const int m = (int)min((int64_t)kDerivedTile, d1 - d);
        for (int b0 = (int)(threadIdx.x >> 6) * rpw; b0 <= m; b0 += 4 * rpw) {
            const int b = b0 + (lane >> l2);
            double x = 0.0;
            if (b <= m) {
                const double* v = src + (d + b) * I.ratio;
                int64_t j = lane & (lpr - 1);
                if (I.ratio >= 8 * 64) {  // long blocks: eight loads in flight per lane
                    double a[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                    for (; j + 7 * 64 < I.ratio; j += 8 * 64)
#pragma unroll
                        for (int u = 0; u < 8; ++u) a[u] = a[u] + v[j + 64 * u];
                    x = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
                }
                for (; j < I.ratio; j += lpr) x = x + v[j];
            }
            for (int off = lpr >> 1; off > 0; off >>= 1) x = x + __shfl_xor(x, off, 64);
            if (b <= m && (lane & (lpr - 1)) == 0) {
                sums[b] = x;
                if (I.store >= 0) ws[I.store + d + b] = x;  // a share's last block is its neighbour's first: the same value
            }
        }
        __syncthreads();
        for (int j = threadIdx.x; j < m; j += 256) s = s + fabs(sums[j + 1] - sums[j]);
        __syncthreads();
    }
    for (int off = 32; off > 0; off >>= 1) s = s + __shfl_xor(s, off, 64);
    if (lane == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) ws[I.part + wb] = (red[0] + red[1]) + (red[2] + red[3]);
}

// score = (sum of the parts of |S[j+1] - S[j]|) / p / (blocks - 1): the parts are one
// value per workgroup of k_score_derived, or the records of a pass, whose units'
// neighbouring sums are compared here.  The last entry is the count of x + eps <= 0.
constexpr int kFinalMax = 64;
struct FinalItem {
    int64_t off;     // parts, or records
    int32_t count;   // parts, or units
    int32_t units;   // 1: records
    double p;        // period (0: a plain sum, the count)
    double ndiff;
};
struct FinalBatch {
    double* ws;
    int64_t stride;
    double* scores[kScoreTensors];
    int32_t first, count;
    FinalItem item[kFinalMax];
};
static_assert(sizeof(FinalBatch) <= 4000, "kernel arguments are limited to 4 KB");

__global__ __launch_bounds__(256) void k_score_final(const FinalBatch B) {
    __shared__ double red[4];
    const FinalItem I = B.item[blockIdx.x];
    const double* __restrict__ v = B.ws + blockIdx.y * B.stride + I.off;
    double s = 0.0;
    for (int i = threadIdx.x; i < I.count; i += 256) {
        s = s + v[i];
        if (I.units && i + 1 < I.count) s = s + fabs(v[I.count + i + 1] - v[2 * (int64_t)I.count + i]);
    }
    for (int off = 32; off > 0; off >>= 1) s = s + __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        s = (red[0] + red[1]) + (red[2] + red[3]);
        B.scores[blockIdx.y][B.first + blockIdx.x] = I.p > 0.0 ? s / I.p / I.ndiff : s;
    }
}

__global__ void k_zero_f64(double* p, int n) {
    const int i = threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// ------------------------------------------------------------------ variance / CoV
template <typename T>
__global__ __launch_bounds__(256) void k_block_var(const T* __restrict__ v, int64_t nblocks, int64_t period,
                                                   int squared, int cov, double* __restrict__ acc) {
    const int lane = threadIdx.x & 63;
    for (int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); blk < nblocks; blk += (int64_t)gridDim.x * 4) {
        const int64_t base = blk * period;
        float sx = 0.0f, sx2 = 0.0f;
        for (int64_t j = lane; j < period; j += 64) {
            const float a = to_f32(v[base + j]);
            const float x = squared ? a : a * a;
            const float x2 = x * x;
            sx = sx + x;
            sx2 = sx2 + x2;
        }
        sx = group_sum(sx, 64);
        sx2 = group_sum(sx2, 64);
        if (lane == 0) {
            const float mean = sx / (float)period;
            float var = sx2 / (float)period;
            const float m2 = mean * mean;
            var = var - m2;
            if (var < 0.0f) var = 0.0f;
            if (!cov) {
                atomicAdd(&acc[0], (double)var);
            } else if (mean < 0.0f) {
                atomicAdd(&acc[2], 1.0);
            } else if (mean > 0.0f) {
                atomicAdd(&acc[0], (double)(sqrtf(var) / mean));
                atomicAdd(&acc[1], 1.0);
            }
        }
    }
}

__global__ void k_var_final(double* acc, int64_t nblocks) { acc[0] = sqrt(acc[0] / (double)nblocks); }

namespace {
int grid_cap(int64_t units) {
    int64_t g = (units + 3) / 4;
    if (g < 1) g = 1;
    if (g > 4096) g = 4096;
    return (int)g;
}

// How the divisors of one tensor size are scored, and its workspace (doubles).
struct PassPlan {
    int q = 0;         // a common multiple of the items' p that divides n; chunks are `times` of it
    int times = 1, chunks_per_unit = 1, nunits = 1;
    int64_t nchunks = 0, rec_off = 0, bad_off = -1;
    std::vector<int> p;             // ascending, p[0] = 1
    std::vector<ScoreItem> item;
};
struct ValueSums { int64_t p, off, bad_off; };  // block sums straight from the values
struct SizePlan {
    std::vector<PassPlan> pass;
    std::vector<ValueSums> value;
    std::vector<DerivedItem> derived[2];
    std::vector<int> derived_wgs[2];
    std::vector<FinalItem> final;   // one per divisor, then the count
    int64_t total = 0;
};

constexpr int64_t kUsefulSource = 6;    // stored sums of at least this many elements: 8 B written and read for each
constexpr int64_t kStageOneMax = 1024;  // longer divisors are read from the first stage's sums where that is much less

// The pass over chunks that takes `need` (a divisor of n, at most kPassMax) and the
// most of the other open divisors up to kPassMax: their least common multiple q
// divides n, and the sums of q elements fit in LDS.
PassPlan choose_pass(int64_t n, int64_t need, const std::vector<int64_t>& divs, const std::vector<char>& open) {
    PassPlan best;
    for (int64_t q = need; q <= kScoreChunk; q += need) {
        if (n % q) continue;
        std::vector<int> list(1, 1);
        int64_t room = kScoreBudget - q;
        if (need > 1) {
            list.push_back((int)need);
            room -= q / need;
        }
        for (size_t d = 0; d < divs.size() && divs[d] <= kPassMax && (int)list.size() < kScoreItems; ++d) {
            const int64_t p = divs[d];
            if (p == 1 || p == need || !open[d] || q % p || q / p > room) continue;
            room -= q / p;
            list.push_back((int)p);
        }
        if (list.size() > best.p.size()) {
            best.q = (int)q;
            best.p = list;
        }
    }
    std::sort(best.p.begin(), best.p.end());
    return best;
}

int make_plan(int64_t n, const int64_t* dv, int ndiv, SizePlan& P) {
    for (int d = 0; d < ndiv; ++d) {
        const int64_t p = dv[d];
        if (p <= 0 || n % p) return fail_inval("divisor %lld does not divide numel %lld", (long long)p, (long long)n);
        if (n / p < 2) return fail_inval("Expected at least two blocks to compare adjacent block means.");
        if (d > 0 && dv[d] <= dv[d - 1]) return fail_inval("divisors must be strictly ascending");
    }
    const std::vector<int64_t> divs(dv, dv + ndiv);
    std::vector<char> open(ndiv, 1);
    auto add_pass = [&](int64_t need) {
        PassPlan pass = choose_pass(n, need, divs, open);
        for (int d = 0; d < ndiv; ++d)
            if (std::find(pass.p.begin(), pass.p.end(), divs[d]) != pass.p.end()) open[d] = 0;
        P.pass.push_back(pass);
    };
    for (int d = 0; d < ndiv && divs[d] <= kPassMax; ++d)
        if (open[d]) add_pass(divs[d]);
    // The others, ascending: each from the longest block sums at hand that it is a
    // multiple of.  Sums of a pass or from the values (stage 0) are read n / q at a
    // time, so long ones from sums that the first stage forms.
    struct Source { int kind; int at; int64_t q; };  // kind 0: a pass's item, 1: values, 2: a derived divisor
    std::vector<Source> from(ndiv, Source{-1, 0, 0});
    for (int d = 0; d < ndiv; ++d) {
        if (!open[d]) continue;
        const int64_t p = divs[d];
        Source best{-1, 0, 0}, late{-1, 0, 0};
        for (size_t k = 0; k < P.pass.size(); ++k)
            for (int q : P.pass[k].p)
                if (p % q == 0 && q > best.q) best = Source{0, (int)k, q};
        for (size_t k = 0; k < P.value.size(); ++k)
            if (p % P.value[k].p == 0 && P.value[k].p > best.q) best = Source{1, (int)k, P.value[k].p};
        for (int e = 0; e < d; ++e)
            if (open[e] && from[e].kind < 2 && p % divs[e] == 0 && divs[e] > late.q) late = Source{2, e, divs[e]};
        if (p > kStageOneMax && late.q >= 8 * std::max<int64_t>(best.q, 1)) best = late;
        if (best.q < kUsefulSource) {
            int64_t part = 1;  // a part of p that a pass can take, if none has
            for (int64_t q = kPassMax; q >= kUsefulSource && part == 1; --q)
                if (p % q == 0) part = q;
            if (part > 1) {
                P.pass.push_back(choose_pass(n, part, divs, open));
                best = Source{0, (int)P.pass.size() - 1, part};
            } else {
                P.value.push_back(ValueSums{p, 0, -1});
                best = Source{1, (int)P.value.size() - 1, p};
            }
        }
        from[d] = best;
    }
    // offsets
    int64_t o = 0;
    auto take = [&](int64_t count) {
        const int64_t at = o;
        o += (count + 31) & ~(int64_t)31;
        return at;
    };
    P.final.resize(ndiv + 1);
    std::vector<char> scored(ndiv, 0);
    for (size_t k = 0; k < P.pass.size(); ++k) {
        PassPlan& pass = P.pass[k];
        // as much of the LDS as leaves about a thousand chunks, or 512 elements each
        int64_t sums = 0;
        for (int p : pass.p) sums += pass.q / p;
        const int64_t aim = std::max<int64_t>(512, n / 1024);
        pass.times = (int)std::max<int64_t>(1, std::min({kScoreBudget / sums, (aim + pass.q - 1) / pass.q, n / pass.q, (int64_t)kScoreChunk / pass.q}));
        const int64_t len = (int64_t)pass.q * pass.times;
        pass.nchunks = (n + len - 1) / len;
        // about a thousand units, of up to 16 chunks
        pass.chunks_per_unit = (int)std::min<int64_t>(16, std::max<int64_t>(1, pass.nchunks / 1024));
        const int64_t units = (pass.nchunks + pass.chunks_per_unit - 1) / pass.chunks_per_unit;
        if (units > INT32_MAX) return fail_inval("tensor too large");
        pass.nunits = (int)units;
        int at = 0, recs = 0;
        for (size_t i = 0; i < pass.p.size(); ++i) {
            const int p = pass.p[i];
            ScoreItem it;
            memset(&it, 0, sizeof(it));
            it.count = (int)(len / p);
            it.tail = (int)((n - (pass.nchunks - 1) * len) / p);
            it.at = at;
            at += it.count;
            it.store = -1;
            it.rec = -1;
            size_t parent = 0;
            for (size_t j = 1; j < i; ++j)
                if (p % pass.p[j] == 0) parent = j;
            if (i > 0) {
                it.parent = pass.item[parent].at;
                it.ratio = p / pass.p[parent];
                it.level = pass.item[parent].level + 1;
            }
            const auto f = std::find(divs.begin(), divs.end(), (int64_t)p);
            if (f != divs.end() && !scored[f - divs.begin()] && !open[f - divs.begin()]) {
                scored[f - divs.begin()] = 1;
                it.rec = recs++;
            }
            pass.item.push_back(it);
        }
        pass.rec_off = take(3 * (int64_t)recs * pass.nunits);
        if (k == 0) pass.bad_off = take(pass.nunits);
        for (size_t i = 0; i < pass.p.size(); ++i) {
            if (pass.item[i].rec < 0) continue;
            const int64_t p = pass.p[i];
            P.final[std::find(divs.begin(), divs.end(), p) - divs.begin()] =
                FinalItem{pass.rec_off + 3 * (int64_t)pass.item[i].rec * pass.nunits, pass.nunits, 1, (double)p,
                          (double)(n / p - 1)};
        }
        // items in level order, so that one barrier serves a level
        std::vector<ScoreItem> sorted = pass.item;
        std::vector<int> order(sorted.size());
        for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
        std::stable_sort(order.begin(), order.end(),
                         [&](int a, int b) { return sorted[a].level < sorted[b].level; });
        std::vector<int> ps = pass.p;
        for (size_t i = 0; i < order.size(); ++i) {
            pass.item[i] = sorted[order[i]];
            pass.p[i] = ps[order[i]];
        }
    }
    for (size_t k = 0; k < P.value.size(); ++k) {
        ValueSums& v = P.value[k];
        v.off = take(n / v.p);
        if (P.pass.empty() && k == 0) v.bad_off = take(n / v.p);
    }
    std::vector<int> slot(ndiv, -1);  // of a first-stage divisor among P.derived[0]
    for (int d = 0; d < ndiv; ++d) {
        if (!open[d]) continue;
        const int64_t p = divs[d], nb = n / p, q = from[d].q;
        const int stage = from[d].kind == 2 ? 1 : 0;
        int64_t* src;
        if (from[d].kind == 0) {
            PassPlan& pass = P.pass[from[d].at];
            src = &pass.item[std::find(pass.p.begin(), pass.p.end(), (int)q) - pass.p.begin()].store;
        } else if (from[d].kind == 1) {
            src = &P.value[from[d].at].off;
        } else {
            src = &P.derived[0][slot[from[d].at]].store;
        }
        if (*src < 0) *src = take(n / q);
        // a workgroup for every 4096 source entries, no more than there are differences
        const int64_t wgs = std::min<int64_t>(std::min<int64_t>(nb - 1, 1024), std::max<int64_t>(1, n / q / 4096));
        const int64_t at = *src;
        if (stage == 0) slot[d] = (int)P.derived[0].size();
        P.derived[stage].push_back(DerivedItem{at, p / q, nb, take(wgs), -1});
        P.derived_wgs[stage].push_back((int)wgs);
        P.final[d] = FinalItem{P.derived[stage].back().part, (int32_t)wgs, 0, (double)p, (double)(nb - 1)};
    }
    if (!P.pass.empty()) P.final[ndiv] = FinalItem{P.pass[0].bad_off, P.pass[0].nunits, 0, 0.0, 0.0};
    else P.final[ndiv] = FinalItem{P.value[0].bad_off, (int32_t)std::min<int64_t>(n / P.value[0].p, INT32_MAX), 0, 0.0, 0.0};
    P.total = o;
    return GEFEN_OK;
}

template <typename T>
void launch_pass(const ScorePass& A, int mode, int ntensors, hipStream_t st) {
    const dim3 grid((unsigned)A.nunits, (unsigned)ntensors), wg(kScoreThreads);
    if (mode == 0) hipLaunchKernelGGL((k_score_pass<T, 0>), grid, wg, 0, st, A);
    else if (mode == 1) hipLaunchKernelGGL((k_score_pass<T, 1>), grid, wg, 0, st, A);
    else hipLaunchKernelGGL((k_score_pass<T, 2>), grid, wg, 0, st, A);
}
template <typename T>
void launch_value_sums(const void* v, int64_t nblocks, int64_t p, int mode, double eps, double* out, double* bad,
                       hipStream_t st) {
    hipLaunchKernelGGL(k_log_block_sums<T>, dim3(grid_cap(nblocks)), dim3(256), 0, st, static_cast<const T*>(v), nblocks,
                       p, mode, eps, out, bad);
}

// The scores of `nt` tensors of one size and dtype, with the workspace of all of them.
int run_scores(const void* const* values, double* const* scores, int nt, int dtype, int64_t n, int ndiv, int mode,
               double eps, double* ws, const SizePlan& P, hipStream_t st) {
    const int64_t stride = P.total;
    for (const PassPlan& pass : P.pass) {
        ScorePass A;
        memset(&A, 0, sizeof(A));
        for (int t = 0; t < nt; ++t) A.values[t] = values[t];
        A.ws = ws;
        A.stride = stride;
        A.nchunks = pass.nchunks;
        A.rec_off = pass.rec_off;
        A.bad_off = pass.bad_off;
        A.eps = eps;
        A.q = pass.item[0].count;
        A.tail = pass.item[0].tail;
        A.nitems = (int)pass.item.size();
        A.chunks_per_unit = pass.chunks_per_unit;
        A.nunits = pass.nunits;
        for (size_t i = 0; i < pass.item.size(); ++i) A.item[i] = pass.item[i];
        if (dtype == GEFEN_F32) launch_pass<float>(A, mode, nt, st);
        else if (dtype == GEFEN_BF16) launch_pass<bf16_t>(A, mode, nt, st);
        else launch_pass<f16_t>(A, mode, nt, st);
        const int rc = launch_status("gefen period pass");
        if (rc) return rc;
    }
    for (const ValueSums& v : P.value)
        for (int t = 0; t < nt; ++t) {
            double* w = ws + t * stride;
            double* bad = v.bad_off >= 0 ? w + v.bad_off : nullptr;
            if (dtype == GEFEN_F32) launch_value_sums<float>(values[t], n / v.p, v.p, mode, eps, w + v.off, bad, st);
            else if (dtype == GEFEN_BF16) launch_value_sums<bf16_t>(values[t], n / v.p, v.p, mode, eps, w + v.off, bad, st);
            else launch_value_sums<f16_t>(values[t], n / v.p, v.p, mode, eps, w + v.off, bad, st);
            const int rc = launch_status("gefen period block sums");
            if (rc) return rc;
        }
    for (int stage = 0; stage < 2; ++stage)
    for (size_t first = 0; first < P.derived[stage].size(); first += kDerivedMax) {
        DerivedBatch B;
        memset(&B, 0, sizeof(B));
        B.ws = ws;
        B.stride = stride;
        B.count = (int)std::min<size_t>(kDerivedMax, P.derived[stage].size() - first);
        int wg = 0;
        for (int i = 0; i < B.count; ++i) {
            B.item[i] = P.derived[stage][first + i];
            B.wg_begin[i] = wg;
            wg += P.derived_wgs[stage][first + i];
        }
        B.wg_begin[B.count] = wg;
        hipLaunchKernelGGL(k_score_derived, dim3((unsigned)wg, (unsigned)nt), dim3(256), 0, st, B);
        const int rc = launch_status("gefen period derived sums");
        if (rc) return rc;
    }
    for (int first = 0; first < ndiv + 1; first += kFinalMax) {
        FinalBatch B;
        memset(&B, 0, sizeof(B));
        B.ws = ws;
        B.stride = stride;
        for (int t = 0; t < nt; ++t) B.scores[t] = scores[t];
        B.first = first;
        B.count = std::min(kFinalMax, ndiv + 1 - first);
        for (int i = 0; i < B.count; ++i) B.item[i] = P.final[first + i];
        hipLaunchKernelGGL(k_score_final, dim3((unsigned)B.count, (unsigned)nt), dim3(256), 0, st, B);
        const int rc = launch_status("gefen period final");
        if (rc) return rc;
    }
    return GEFEN_OK;
}

// Tensors of one launch: their workspaces together stay small, for it is reused
// from launch to launch.
int tensors_per_launch(const SizePlan& P) {
    const int64_t fit = ((int64_t)64 << 20) / std::max<int64_t>(1, P.total * (int64_t)sizeof(double));
    return (int)std::min<int64_t>(kScoreTensors, std::max<int64_t>(1, fit));
}

int check_values(const void* v, int dt, int64_t n, int64_t period) {
    if (!valid_dtype(dt)) return fail_inval("Expected a floating-point tensor.");
    if (period <= 0) return fail_inval("Expected a positive period.");
    if (n <= 0) return fail_inval("Expected a non-empty tensor.");
    if (n % period) return fail_inval("Expected tensor length to be divisible by period.");
    if (!v) return fail_inval("null values pointer");
    return GEFEN_OK;
}
}  // namespace
}  // namespace gefen

using namespace gefen;

extern "C" size_t gefen_period_scores_workspace_size(int64_t numel, const int64_t* divs, int ndiv) {
    if (numel <= 0 || ndiv <= 0 || !divs) return 0;
    SizePlan P;
    if (make_plan(numel, divs, ndiv, P)) return 0;
    return (size_t)P.total * sizeof(double);
}

extern "C" int gefen_period_scores(const void* values, int dtype, int64_t numel, const int64_t* divs, int ndiv,
                                   int mode, double epsilon, double* scores, void* workspace,
                                   gefen_stream_t stream) {
    if (ndiv <= 0 || !divs) return fail_inval("no divisors");
    int rc = check_values(values, dtype, numel, 1);
    if (rc) return rc;
    if (mode < 0 || mode > 2) return fail_inval("invalid mode %d", mode);
    if (!scores || !workspace) return fail_inval("null pointer");
    SizePlan P;
    rc = make_plan(numel, divs, ndiv, P);
    if (rc) return rc;
    return run_scores(&values, &scores, 1, dtype, numel, ndiv, mode, epsilon, static_cast<double*>(workspace), P,
                      reinterpret_cast<hipStream_t>(stream));
}

namespace gefen {
namespace {
// Groups of tasks that share size, dtype and divisors.
struct TaskGroup {
    std::vector<int> at;
    SizePlan plan;
};
int group_tasks(const gefen_period_task* tasks, int ntasks, std::vector<TaskGroup>& groups) {
    for (int i = 0; i < ntasks; ++i) {
        const gefen_period_task& t = tasks[i];
        if (t.ndiv <= 0 || !t.divs) return fail_inval("no divisors");
        int rc = check_values(t.values, t.dtype, t.numel, 1);
        if (rc) return rc;
        if (!t.scores) return fail_inval("null pointer");
        TaskGroup* g = nullptr;
        for (TaskGroup& o : groups) {
            const gefen_period_task& r = tasks[o.at[0]];
            if (r.numel == t.numel && r.dtype == t.dtype && r.ndiv == t.ndiv &&
                memcmp(r.divs, t.divs, sizeof(int64_t) * (size_t)t.ndiv) == 0) {
                g = &o;
                break;
            }
        }
        if (!g) {
            groups.emplace_back();
            g = &groups.back();
            rc = make_plan(t.numel, t.divs, t.ndiv, g->plan);
            if (rc) return rc;
        }
        g->at.push_back(i);
    }
    return GEFEN_OK;
}
}  // namespace
}  // namespace gefen

extern "C" size_t gefen_period_scores_tasks_workspace_size(const gefen_period_task* tasks, int ntasks) {
    if (!tasks || ntasks <= 0) return 0;
    std::vector<TaskGroup> groups;
    if (group_tasks(tasks, ntasks, groups)) return 0;
    int64_t most = 0;
    for (const TaskGroup& g : groups)
        most = std::max(most, g.plan.total * std::min<int64_t>(tensors_per_launch(g.plan), (int64_t)g.at.size()));
    return (size_t)most * sizeof(double);
}

extern "C" int gefen_period_scores_tasks(const gefen_period_task* tasks, int ntasks, int mode, double epsilon,
                                         void* workspace, gefen_stream_t stream) {
    if (ntasks < 0 || (ntasks > 0 && !tasks)) return fail_inval("invalid task array");
    if (ntasks == 0) return GEFEN_OK;
    if (mode < 0 || mode > 2) return fail_inval("invalid mode %d", mode);
    if (!workspace) return fail_inval("null pointer");
    std::vector<TaskGroup> groups;
    int rc = group_tasks(tasks, ntasks, groups);
    if (rc) return rc;
    for (const TaskGroup& g : groups) {
        const int step = tensors_per_launch(g.plan);
        for (size_t first = 0; first < g.at.size(); first += step) {
            const int nt = (int)std::min<size_t>(step, g.at.size() - first);
            const void* values[kScoreTensors];
            double* scores[kScoreTensors];
            for (int i = 0; i < nt; ++i) {
                values[i] = tasks[g.at[first + i]].values;
                scores[i] = tasks[g.at[first + i]].scores;
            }
            const gefen_period_task& t = tasks[g.at[0]];
            rc = run_scores(values, scores, nt, t.dtype, t.numel, t.ndiv, mode, epsilon, static_cast<double*>(workspace),
                            g.plan, reinterpret_cast<hipStream_t>(stream));
            if (rc) return rc;
        }
    }
    return GEFEN_OK;
}

extern "C" int gefen_average_adjacent_log_block_mean_difference(const void* values, int dtype, int64_t numel,
                                                                int64_t period, int input_is_squared,
                                                                double epsilon, double* out,
                                                                gefen_stream_t stream) {
    int rc = check_values(values, dtype, numel, period);
    if (rc) return rc;
    if (!(epsilon > 0.0)) return fail_inval("Expected a positive epsilon.");
    if (numel / period < 2) return fail_inval("Expected at least two blocks to compare adjacent block means.");
    if (!out) return fail_inval("null output pointer");
    const int64_t divs[1] = {period};
    SizePlan P;
    rc = make_plan(numel, divs, 1, P);
    if (rc) return rc;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    void* ws = nullptr;
    hipError_t e = device_malloc_async(&ws, (size_t)P.total * sizeof(double), st);
    if (e != hipSuccess) return hip_status(e, "hipMallocAsync(period workspace)");
    rc = run_scores(&values, &out, 1, dtype, numel, 1, input_is_squared ? 0 : 2, epsilon, static_cast<double*>(ws), P,
                    st);
    (void)hipFreeAsync(ws, st);
    return rc;
}

static int block_var_common(const void* values, int dtype, int64_t numel, int64_t period, int squared, double* out,
                            int cov, gefen_stream_t stream) {
    int rc = check_values(values, dtype, numel, period);
    if (rc) return rc;
    if (!out) return fail_inval("null output pointer");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_zero_f64, dim3(1), dim3(64), 0, st, out, cov ? 3 : 1);
    rc = launch_status("gefen block variance zero");
    if (rc) return rc;
    const int64_t nb = numel / period;
    const int grid = grid_cap(nb);
    if (dtype == GEFEN_F32)
        hipLaunchKernelGGL(k_block_var<float>, dim3(grid), dim3(256), 0, st, static_cast<const float*>(values), nb,
                           period, squared, cov, out);
    else if (dtype == GEFEN_BF16)
        hipLaunchKernelGGL(k_block_var<bf16_t>, dim3(grid), dim3(256), 0, st, static_cast<const bf16_t*>(values), nb,
                           period, squared, cov, out);
    else
        hipLaunchKernelGGL(k_block_var<f16_t>, dim3(grid), dim3(256), 0, st, static_cast<const f16_t*>(values), nb,
                           period, squared, cov, out);
    rc = launch_status("gefen block variance");
    if (rc || cov) return rc;
    hipLaunchKernelGGL(k_var_final, dim3(1), dim3(1), 0, st, out, nb);
    return launch_status("gefen block variance final");
}

extern "C" int gefen_average_within_block_variance(const void* values, int dtype, int64_t numel, int64_t period,
                                                   int input_is_squared, double* out, gefen_stream_t stream) {
    return block_var_common(values, dtype, numel, period, input_is_squared, out, 0, stream);
}

extern "C" int gefen_average_within_block_coefficient_of_variation(const void* values, int dtype, int64_t numel,
                                                                   int64_t period, int input_is_squared,
                                                                   double* out, gefen_stream_t stream) {
    return block_var_common(values, dtype, numel, period, input_is_squared, out, 1, stream);
}
