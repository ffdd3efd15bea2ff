// gemm_tiles.h — what the prefill GEMM's plans (gemm_rpl.hip) and its tile
// kernels (gemm_tiles.hip) share.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "wv_internal.h"

namespace wv {

struct GemmArgs {
    RplArgs w;
    // fp16 8-column blocks of X in permuted k order, row m scaled by
    // 1 / xscale[m]: [M][K/8] row-major, or for k_gemm_rg in MFMA A-fragment
    // order [K/16][ceil(M/32)][64] (lane l of fragment (q, tile): token
    // 32*tile + l%32, block 2q + l/32; tokens past M are zero)
    const uint4* xh;
    const float* xscale;   // [M] power-of-two factor of each row's fp16 copy
    float* y;         // [M][rows] (splits == 1) or partials [split][M][rows]
    int M, K;
    int sb_per_split;
};

enum { GEMM_PW = 1, GEMM_RG = 2 };
// k_gemm_rg waves per block: 8 (2 per SIMD) for one or two 32-token tiles,
// 4 (1 per SIMD) for four.
constexpr int rg_waves(int tm) { return tm == 4 ? 4 : 8; }
struct GemmPlan {
    int kind, bm, splits, sb_per_split, W, per;
};

// gemm_tiles.hip is compiled once per part, each with the kernels that
// gemm_part gives it (rpl_operands.h): the compiler takes up to a minute for an
// instance of k_gemm_q4k_pw whose instructions are spread by hand, and one file
// of all of them took it nine.
constexpr int kGemmParts = 8;
template <int PART>
int launch_gemm_tiles(const DevBlob& b, const GemmPlan& p, dim3 grid, hipStream_t s, const GemmArgs& ga);

}  // namespace wv
