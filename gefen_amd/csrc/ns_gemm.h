// The tiled batched GEMM of the Newton-Schulz products (ns_gemm.hip), as the
// entry points and the Newton-Schulz driver (newton_schulz.hip) launch it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "capi_internal.h"

namespace gefen {
namespace ns {

constexpr int kTileUnit = 128;  // sides of every product are multiples of the smaller tile
constexpr int kStepK = 64;      // and its contraction length of the K step

// C_b = alpha * A_b @ B_b^T + beta * D_b for b < batch (see ns_gemm.hip).
struct TileGemm {
    const uint16_t* A;
    const uint16_t* B;
    uint16_t* C;
    uint16_t* CT;
    const uint16_t* D;
    int64_t lda, ldb, ldc, ldct, ldd;
    int64_t sa, sb, sc, sct, sd;  // batch strides (elements)
    int M, N, K;
    float alpha, beta;
    int tiles_n;   // N / T
    int tiles;     // tiles per matrix
    int symmetric;
    int d_t;       // D is given as D^T [N, M] (row stride ldd): four rows of one column are one 8-byte load
    int vm, vn;    // rows and columns of the parameter a fused update applies to (M, N without padding)
};

// Estimated microseconds of one product of `batch` matrices with the better tile
// (small: which one that is).
double product_us(int m, int n, int k, bool symmetric, int batch, bool* small);

// The product of every matrix (mn: both operands MN-major, the Gram product from
// X^T).  Sides multiples of kTileUnit, K of kStepK, operands checked by the caller.
int launch_product(TileGemm g, int batch, bool mn, hipStream_t st, const char* what);

// The product applied as GefenMuon's update of tasks[0 .. batch): tasks share a
// dtype and orientation and have been checked.  edge: g.vm x g.vn parameters that
// end inside a tile or are not 8-element aligned.
int launch_product_apply(TileGemm g, int batch, const gefen_muon_apply_task* tasks, bool edge, hipStream_t st,
                         const char* what);

}  // namespace ns
}  // namespace gefen
