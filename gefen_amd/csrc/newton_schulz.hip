// Newton-Schulz orthogonalisation (gefen_muon.py:16-51) of a stack of same-shaped
// matrices of any size, and GefenMuon's update of their parameters, in one call.
//
// The tiled products (ns_gemm.hip) need sides that are multiples of a tile; other
// matrices are zero-padded on the way through the normalisation, which has to
// rewrite the stack anyway.  Zero rows and columns stay zero through X X^T,
// b A + c A A and a X + B X, and add exact zeros at the end of every element's K
// sum, so the valid part equals the unpadded products bit for bit.  The last
// product's epilogue updates the parameters and drops the padding.
#include <math.h>
#include <string.h>

#include <algorithm>

#include "capi_internal.h"
#include "common.h"
#include "ns_gemm.h"

namespace gefen {
namespace ns {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Reciprocal (float64) of matrix g's divisor max(bf16(||x||), bf16(eps)), from its
// sum of squares (gefen_ns_prepare_sumsq).
__device__ __forceinline__ double inverse_norm(const double* sumsq, const int32_t* index, int g, float eps_bf16) {
    const double* slots = sumsq + (size_t)(index ? index[g] : g) * GEFEN_SUMSQ_STRIDE;
    double s = 0.0;
    for (int i = 0; i < GEFEN_SUMSQ_SLOTS; ++i) s += slots[16 * i];
    const float nrm = round_to<bf16_t>((float)sqrt(s));
    return 1.0 / (double)((nrm < eps_bf16) ? eps_bf16 : nrm);
}

// Eight elements of a row from column c, zeros past column `cols`.
__device__ __forceinline__ AnyVec<bf16_t, 8> row_chunk(const bf16_t* row, int c, int cols) {
    if (c + 8 <= cols) return *reinterpret_cast<const AnyVec<bf16_t, 8>*>(row + c);
    AnyVec<bf16_t, 8> v;
#pragma unroll
    for (int u = 0; u < 8; ++u) v.v[u] = c + u < cols ? row[c + u] : bf16_t{0};
    return v;
}

// The same quotient as k_scale_transpose forms it: the float64 product with the
// reciprocal rounded to float (div_by_block), then to bf16.
__device__ __forceinline__ uint32_t scaled_bits(bf16_t v, double rd) {
    return from_f32<bf16_t>(div_by_block(to_f32(v), rd)).bits;
}

// out[g] [out_rows, out_cols] = x[g] / d_g, zero-padded; x[g] [rows, cols] tight.
// Eight output elements per thread; traffic-bound (2 B read, 2 B written).
__global__ __launch_bounds__(256) void k_pad_scale(const bf16_t* __restrict__ x, uint16_t* __restrict__ out, int rows,
                                                   int cols, int out_rows, int out_cols,
                                                   const double* __restrict__ sumsq, const int32_t* __restrict__ index,
                                                   float eps_bf16) {
    const int g = blockIdx.y;
    const int chunks = out_cols / 8;
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= (int64_t)out_rows * chunks) return;
    const int r = (int)(q / chunks), c = (int)(q % chunks) * 8;
    u32x4 o = {0u, 0u, 0u, 0u};
    if (r < rows && c < cols) {
        const double rd = inverse_norm(sumsq, index, g, eps_bf16);
        const AnyVec<bf16_t, 8> v = row_chunk(x + ((int64_t)g * rows + r) * cols, c, cols);
#pragma unroll
        for (int u = 0; u < 4; ++u) o[u] = scaled_bits(v.v[2 * u], rd) | (scaled_bits(v.v[2 * u + 1], rd) << 16);
    }
    *reinterpret_cast<u32x4*>(out + (int64_t)g * out_rows * out_cols + q * 8) = o;
}

// out[g] [out_rows, out_cols] = (x[g] / d_g)^T, zero-padded: a 64 x 64 tile of the
// output per workgroup, transposed through LDS as in k_scale_transpose.
constexpr int kPadTile = 64;
__global__ __launch_bounds__(256) void k_pad_scale_transpose(const bf16_t* __restrict__ x, uint16_t* __restrict__ out,
                                                             int rows, int cols, int out_rows, int out_cols,
                                                             const double* __restrict__ sumsq,
                                                             const int32_t* __restrict__ index, float eps_bf16) {
    __shared__ uint16_t tile[kPadTile][kPadTile + 2];
    const int g = blockIdx.z;
    const int r0 = blockIdx.y * kPadTile, c0 = blockIdx.x * kPadTile;  // rows and columns of x
    const int t = threadIdx.x;
    const double rd = inverse_norm(sumsq, index, g, eps_bf16);
    const int r = t >> 2, cc = (t & 3) * 16;
    const bf16_t* row = x + ((int64_t)g * rows + min(r0 + r, rows - 1)) * cols;
    const int lim = r0 + r < rows ? cols : 0;
    AnyVec<bf16_t, 8> v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) v[h] = row_chunk(row, c0 + cc + 8 * h, lim);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int u = 0; u < 8; ++u) tile[r][cc + 8 * h + u] = (uint16_t)scaled_bits(v[h].v[u], rd);
    __syncthreads();
    const int c = t >> 2, rr = (t & 3) * 16;
    uint16_t* q = out + (int64_t)g * out_rows * out_cols + (int64_t)(c0 + c) * out_cols + r0 + rr;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        u32x4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            o[k] = (uint32_t)tile[rr + 8 * h + 2 * k][c] | ((uint32_t)tile[rr + 8 * h + 2 * k + 1][c] << 16);
        *reinterpret_cast<u32x4*>(q + 8 * h) = o;
    }
}

// Padded sides [mp, np] of X [m, n] (m <= n) and the layout of the work buffers:
// X^T twice [np, mp], and two Gram-sized buffers [mp, mp], per matrix.
struct PadPlan {
    int m, n, mp, np;
    size_t xt, t1, gram, upd, total;  // byte offsets
};

int64_t round_up(int64_t v, int64_t unit) { return (v + unit - 1) / unit * unit; }

PadPlan pad_plan(int batch, int rows, int cols) {
    PadPlan p;
    p.m = std::min(rows, cols);
    p.n = std::max(rows, cols);
    // the multiple of 128 or 256 for which the three products of an iteration are
    // estimated faster: 256 where it adds little padding and lets full chips of
    // workgroups take the larger tile
    double best = 0.0;
    for (int unit : {kTileUnit, 2 * kTileUnit}) {
        const int mp = (int)round_up(p.m, unit), np = (int)round_up(p.n, unit);
        bool small;
        const double us = product_us(mp, mp, np, true, batch, &small) + product_us(mp, mp, mp, true, batch, &small) +
                          product_us(mp, np, mp, false, batch, &small);
        if (unit == kTileUnit || us < best) {
            best = us;
            p.mp = mp;
            p.np = np;
        }
    }
    const size_t x = round_up((int64_t)batch * p.mp * p.np * 2, 256), a = round_up((int64_t)batch * p.mp * p.mp * 2, 256);
    p.xt = 0;
    p.t1 = x;
    p.gram = 2 * x;
    p.upd = 2 * x + a;
    p.total = 2 * (x + a);
    return p;
}

bool pad_size_ok(int rows, int cols) {
    // a padded matrix is read through a buffer of less than 2^31 bytes
    return round_up(rows, 2 * kTileUnit) * round_up(cols, 2 * kTileUnit) * 2 <= INT32_MAX;
}

}  // namespace ns
}  // namespace gefen

using namespace gefen;

extern "C" size_t gefen_newton_schulz_workspace_size(int batch, int rows, int cols) {
    if (batch <= 0 || rows <= 0 || cols <= 0 || !ns::pad_size_ok(rows, cols)) return 0;
    return ns::pad_plan(batch, rows, cols).total;
}

extern "C" int gefen_newton_schulz_apply(const void* x, int batch, int rows, int cols, double a, double b, double c,
                                         int steps, double eps, const double* sumsq, const int32_t* index,
                                         void* workspace, const gefen_muon_apply_task* tasks, gefen_stream_t stream) {
    if (batch < 0 || rows < 0 || cols < 0) return fail_inval("negative size");
    if (batch == 0 || rows == 0 || cols == 0) return GEFEN_OK;
    if (steps <= 0) return fail_inval("a fused update needs at least one Newton-Schulz step");
    if (!x || !sumsq || !workspace || !tasks) return fail_inval("null pointer");
    if (!ns::pad_size_ok(rows, cols)) return fail_inval("matrix of %d x %d too large for the padded products", rows, cols);
    if (batch > 65535) return fail_inval("batch too large");
    if (!aligned(x, 2) || !aligned(workspace, 16)) return fail_inval("misaligned Newton-Schulz buffer");
    const bool tall = rows > cols;
    const int dt = tasks[0].param_dtype;
    if (!valid_dtype(dt)) return fail_inval("unsupported parameter dtype %d", dt);
    bool edge = false;
    for (int i = 0; i < batch; ++i) {
        const gefen_muon_apply_task& t = tasks[i];
        if (t.param_dtype != dt) return fail_inval("the parameters of one call must share a dtype");
        if ((t.transposed != 0) != tall) return fail_inval("parameter %d is not in the stack's orientation", i);
        if (t.numel != (int64_t)rows * cols)
            return fail_inval("parameter %d has %lld elements, the matrix %lld", i, (long long)t.numel,
                              (long long)rows * cols);
        if (!t.p) return fail_inval("null parameter pointer");
        if (!aligned(t.p, dtype_size(dt))) return fail_inval("misaligned parameter pointer");
        edge = edge || !aligned(t.p, 8 * dtype_size(dt));
    }
    const ns::PadPlan P = ns::pad_plan(batch, rows, cols);
    edge = edge || P.m != P.mp || P.n != P.np;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    uint16_t* xt = reinterpret_cast<uint16_t*>(ws + P.xt);
    uint16_t* t1 = reinterpret_cast<uint16_t*>(ws + P.t1);
    uint16_t* gram = reinterpret_cast<uint16_t*>(ws + P.gram);
    uint16_t* upd = reinterpret_cast<uint16_t*>(ws + P.upd);
    float eps_bf16 = (float)eps;
    {
        uint32_t u;
        memcpy(&u, &eps_bf16, 4);
        u = (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
        memcpy(&eps_bf16, &u, 4);
    }
    // X^T [np, mp]: the stack itself for tall matrices, its transpose otherwise
    if (tall) {
        const int64_t chunks = (int64_t)P.np * P.mp / 8;
        hipLaunchKernelGGL(ns::k_pad_scale, dim3((unsigned)((chunks + 255) / 256), batch), dim3(256), 0, st,
                           static_cast<const bf16_t*>(x), xt, rows, cols, P.np, P.mp, sumsq, index, eps_bf16);
    } else {
        hipLaunchKernelGGL(ns::k_pad_scale_transpose, dim3(P.np / ns::kPadTile, P.mp / ns::kPadTile, batch), dim3(256),
                           0, st, static_cast<const bf16_t*>(x), xt, rows, cols, P.np, P.mp, sumsq, index, eps_bf16);
    }
    int rc = launch_status("gefen_newton_schulz_apply (normalise)");
    const int64_t sx = (int64_t)P.np * P.mp, sg = (int64_t)P.mp * P.mp;
    for (int it = 0; it < steps && rc == GEFEN_OK; ++it) {
        ns::TileGemm g;
        memset(&g, 0, sizeof(g));  // A = X X^T
        g.A = g.B = xt;
        g.C = gram;
        g.lda = g.ldb = g.ldc = P.mp;
        g.sa = g.sb = sx;
        g.sc = sg;
        g.M = g.N = P.mp;
        g.K = P.np;
        g.alpha = 1.0f;
        g.symmetric = 1;
        rc = ns::launch_product(g, batch, true, st, "gefen_newton_schulz_apply (gram)");
        if (rc) break;
        memset(&g, 0, sizeof(g));  // b A + c A A
        g.A = g.B = g.D = gram;
        g.C = upd;
        g.lda = g.ldb = g.ldc = g.ldd = P.mp;
        g.sa = g.sb = g.sc = g.sd = sg;
        g.M = g.N = g.K = P.mp;
        g.alpha = (float)c;
        g.beta = (float)b;
        g.symmetric = g.d_t = 1;
        rc = ns::launch_product(g, batch, false, st, "gefen_newton_schulz_apply (poly)");
        if (rc) break;
        memset(&g, 0, sizeof(g));  // (a X + B X)^T, or the update from it
        g.A = upd;
        g.B = g.D = xt;
        g.lda = g.ldb = g.ldd = g.ldct = P.mp;
        g.sa = sg;
        g.sb = g.sd = g.sct = sx;
        g.M = P.mp;
        g.N = P.np;
        g.K = P.mp;
        g.vm = P.m;
        g.vn = P.n;
        g.alpha = 1.0f;
        g.beta = (float)a;
        g.d_t = 1;
        if (it + 1 < steps) {
            g.CT = t1;
            rc = ns::launch_product(g, batch, false, st, "gefen_newton_schulz_apply (update)");
            std::swap(xt, t1);
        } else {
            rc = ns::launch_product_apply(g, batch, tasks, edge, st, "gefen_newton_schulz_apply (apply)");
        }
    }
    return rc;
}
