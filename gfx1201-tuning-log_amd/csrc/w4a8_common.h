// Operands and tile order shared by the MXFP4 x fp8 GEMM kernels (w4a8_gemm.hip, w4a8_slice.hip).
#pragma once
#include "fp8kv_common.h"
#include <utility>

namespace fp8kv {
namespace w4a8_detail {

constexpr int kBK = 128;                              // k per step: one block-scaled MFMA
constexpr int kXcds = 8;

typedef int v8i __attribute__((ext_vector_type(8)));

__device__ __forceinline__ v8i concat8(u32x4_t lo, u32x4_t hi)
{
    return (v8i){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
}

struct Params {
    const uint8_t* W;
    const uint8_t* St;
    const uint8_t* Xq;
    const uint8_t* Sx;
    __bf16* Out;
    const float* tok_scale;   // per-token mode: fp32 scale of each activation row (Sx unused)
    int N, K, M;
    int nblk, mblk;
    int gm, gn;          // tile order: the 8 XCDs split the token blocks gm ways and the weight blocks gn ways
};

// Tile of workgroup L, or false when L has none.  Workgroup L runs on XCD L % 8 (round-robin
// dispatch); XCD x = (xm, xn) takes token blocks xm, xm + gm, ... and the xn-th range of weight
// blocks, weight-block major, so each XCD's L2 holds its share of the activations and the
// weight tiles it streams are shared by the workgroups running it at the same time.
__device__ __forceinline__ bool tile_of(const Params& P, int L, int& nb, int& mb)
{
    const int x = L % kXcds, slot = L / kXcds;
    const int xm = x % P.gm, xn = x / P.gm;
    const int my_m = (P.mblk - xm + P.gm - 1) / P.gm;
    const int nper = (P.nblk + P.gn - 1) / P.gn;
    const int n_lo = xn * nper;
    const int n_hi = n_lo + nper < P.nblk ? n_lo + nper : P.nblk;
    if (my_m <= 0 || n_lo >= n_hi || slot >= my_m * (n_hi - n_lo)) return false;
    nb = n_lo + slot / my_m;
    mb = xm + P.gm * (slot % my_m);
    return true;
}

// Tiles of the K-splitting kernel (w4a8_slice.hip): 16 tn weight rows x 16 tm tokens, `waves` waves; in
// the order in which the planner tries them.
struct SliceShape {
    int tn, tm, waves;
};
constexpr SliceShape kSliceShapes[] = {{1, 1, 8}, {1, 2, 8}, {2, 1, 8}, {2, 2, 8}, {2, 3, 8}, {2, 4, 8}, {4, 3, 8}, {4, 4, 4}, {4, 8, 4}, {8, 4, 4}};
constexpr int kNumSliceShapes = sizeof(kSliceShapes) / sizeof(kSliceShapes[0]);
constexpr int kSliceMinK = 512;                       // a scale load takes four steps of a row

void launch_slice(int shape, bool tok, dim3 grid, hipStream_t st, const Params& P);

}  // namespace w4a8_detail
}  // namespace fp8kv
