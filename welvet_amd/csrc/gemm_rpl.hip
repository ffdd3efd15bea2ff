// gemm_rpl.hip — batched prefill on the row-interleaved layouts:
// Y[M][rows] = X[M][cols] * W^T with fp16 MFMA (v_mfma_f32_32x32x16_f16) and
// f32 accumulation. It replaces welvet's M independent GEMVs for a token block
// (forwardSIMDBlockFused, layers/dense/simd_block.go:17-39), within the 2e-3
// tolerance of an fp16 contraction.
//
// X is first converted once to fp16 (k_x_f16r), so the GEMM streams half the
// bytes for the operand every row tile re-reads and spends no VALU on it. Each
// token row is scaled by a power of two that puts its max|x| in [2^14, 2^15)
// before the cast, and the epilogue multiplies the row back: the scaling is
// exact, so rows that fit fp16 get the same fp16 values as an unscaled cast,
// while outlier rows (|x| > 65504) stay finite and rows of tiny activations
// keep their precision instead of going subnormal. Weight rows get the same
// treatment from a power-of-two factor stored per row at upload
// (RplArgs::wrow) that puts the row's largest fp16 B-operand value in
// [2^12, 2^13): the B-operand builders multiply the row's scales and mins by
// it before their fp16 cast and the epilogue divides it back out, so rows of
// tiny weights keep fp16's precision and rows past 65504 stay finite.
//
// W goes from the row-interleaved planes straight into MFMA B operands: a
// lane holds 32 columns of its row per chunk, and a lane swap puts them into
// the 32x32x16 operand layout (per-format B-operand builders). Within every
// 8-column block both operands are in k order [0,2,4,6,1,3,5,7], the order in
// which the code spread produces pairs; a dot product over the block does not
// depend on the order. Two kernels (gemm_tiles.hip):
//   * k_gemm_rg, up to 128 tokens: a block per 64-row group, its waves
//     splitting K and reading X fragments straight from global memory, every
//     weight dequantized once;
//   * k_gemm_q4k_pw, more tokens: 256-row x 128- or 256-token tiles with X
//     staged through LDS.
// K is split over gridDim.z when the tile grid alone would leave CUs idle;
// the splits' partials meet in a fixed-order sum.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "gemm_tiles.h"
#include "rpl_operands.h"
#include "wave_ops.h"
#include "wv_internal.h"

namespace wv {
namespace {

// 8 columns of X times `up`, as fp16 pairs in k order [0,2,4,6,1,3,5,7].
__device__ __forceinline__ uint4 pack_x8(float4 lo, float4 hi, float up) {
    lo = make_float4(lo.x * up, lo.y * up, lo.z * up, lo.w * up);
    hi = make_float4(hi.x * up, hi.y * up, hi.z * up, hi.w * up);
    return make_uint4(pack_h2(lo.x, lo.z), pack_h2(hi.x, hi.z), pack_h2(lo.y, lo.w), pack_h2(hi.y, hi.w));
}
__device__ __forceinline__ float absmax8(float4 lo, float4 hi) {
    return fmaxf(fmaxf(fmaxf(fabsf(lo.x), fabsf(lo.y)), fmaxf(fabsf(lo.z), fabsf(lo.w))),
                 fmaxf(fmaxf(fabsf(hi.x), fabsf(hi.y)), fmaxf(fabsf(hi.z), fabsf(hi.w))));
}
// The row's factor from its max|x| (the block-wide reduction), 2^-shift.
__device__ __forceinline__ float row_shift_up(float mx, float* red, float* xscale_m, int t) {
    mx = wave_maximum(mx);
    if ((t & 63) == 0) red[t >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int sh = 0;  // x is multiplied by 2^sh
    if (mx > 0.f && mx <= 3.4028235e38f) sh = min(126, max(-126, 14 - ilogbf(mx)));
    if (t == 0) *xscale_m = ldexpf(1.0f, -sh);
    return ldexpf(1.0f, sh);
}
// silu(g) * u of one element, the expression of the SwiGLU kernels
// (layers/swiglu/cpu.go:41-53).
__device__ __forceinline__ float silu_mul1(float g, float u) { return g / (1.0f + expf(-g)) * u; }
__device__ __forceinline__ float4 silu_mul4(float4 g, float4 u) {
    return make_float4(silu_mul1(g.x, u.x), silu_mul1(g.y, u.y), silu_mul1(g.z, u.z), silu_mul1(g.w, u.w));
}

// X f32 [M][K] -> fp16 blocks of 8 in the B operands' k order
// [0,2,4,6,1,3,5,7] (pack_x8), one block per token row:
// the row's max|x| picks xscale = 2^e with max|x| / xscale in [2^14, 2^15)
// (1 for an all-zero or non-finite row), and the blocks hold x / xscale.
// A row of up to 256 * NR blocks of 8 is read once, into registers, with every
// load issued before the first use (slots past the row re-read its last block).
// FRAG writes the A-fragment order of GemmArgs::xh (block i of row m at
// ((i/2)*mt + m/32)*64 + m%32 + 32*(i%2)); its grid covers the padded rows,
// which get zeros. SW: x is the gate and u the up projection, and the row
// converted is silu(x) * u (the SwiGLU product feeding the down projection).
template <int NR, bool FRAG, bool SW>
__global__ void __launch_bounds__(256) k_x_f16r(const float4* __restrict__ x, const float4* __restrict__ u,
                                                 uint4* __restrict__ xh, float* __restrict__ xscale, int kb8, int M) {
    __shared__ float red[4];
    const int m = blockIdx.x, t = threadIdx.x;
    const int mt = (M + 31) / 32;
    auto put = [&](int i, uint4 v) {
        if constexpr (FRAG)
            xh[(int64_t(i >> 1) * mt + (m >> 5)) * 64 + (m & 31) + 32 * (i & 1)] = v;
        else
            xh[int64_t(m) * kb8 + i] = v;
    };
    if (FRAG && m >= M) {
        for (int i = t; i < kb8; i += 256) put(i, make_uint4(0u, 0u, 0u, 0u));
        return;
    }
    const float4* xr = x + int64_t(m) * kb8 * 2;
    const float4* ur = SW ? u + int64_t(m) * kb8 * 2 : nullptr;
    auto ld = [&](int k) { return SW ? silu_mul4(xr[k], ur[k]) : xr[k]; };
    float mx = 0.f;
    if constexpr (NR > 0) {
        float4 lo[NR], hi[NR];
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const int i = min(t + 256 * j, kb8 - 1);
            lo[j] = xr[2 * i];
            hi[j] = xr[2 * i + 1];
        }
        if constexpr (SW) {
            float4 ul[NR], uh[NR];
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int i = min(t + 256 * j, kb8 - 1);
                ul[j] = ur[2 * i];
                uh[j] = ur[2 * i + 1];
            }
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                lo[j] = silu_mul4(lo[j], ul[j]);
                hi[j] = silu_mul4(hi[j], uh[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < NR; ++j) mx = fmaxf(mx, absmax8(lo[j], hi[j]));
        const float up = row_shift_up(mx, red, xscale + m, t);
#pragma unroll
        for (int j = 0; j < NR; ++j)
            if (t + 256 * j < kb8) put(t + 256 * j, pack_x8(lo[j], hi[j], up));
    } else {  // longer rows: two passes, the second mostly from L2
        for (int i = t; i < kb8; i += 256) mx = fmaxf(mx, absmax8(ld(2 * i), ld(2 * i + 1)));
        const float up = row_shift_up(mx, red, xscale + m, t);
        for (int i = t; i < kb8; i += 256) put(i, pack_x8(ld(2 * i), ld(2 * i + 1), up));
    }
}
// The key-split prompt attention's merge straight into the O projection's
// fp16 operand: per row and head, sum_z 2^(m_z - M) o_z / sum_z 2^(m_z - M) l_z
// over the ks ranges of part ([ks][M][heads][hd + 4]: the unnormalized
// output, then the running max in log2 units and the running sum; ranges
// with m_z = -inf count 0), in the order and arithmetic of the decoder's
// k_attn_prefill_merge, then the row factor and blocks as k_x_f16r<NR, FRAG,
// false> makes them from the merged rows. Every range's values of a slot are
// loaded before the first add.
template <int NR, bool FRAG>
__global__ void __launch_bounds__(256) k_merge_x_f16r(const float* __restrict__ part, int ks, int n_heads, int hd,
                                                       uint4* __restrict__ xh, float* __restrict__ xscale, int kb8,
                                                       int M) {
    constexpr int KS = 8;
    __shared__ float red[4];
    const int m = blockIdx.x, t = threadIdx.x;
    const int mt = (M + 31) / 32;
    auto put = [&](int i, uint4 v) {
        if constexpr (FRAG)
            xh[(int64_t(i >> 1) * mt + (m >> 5)) * 64 + (m & 31) + 32 * (i & 1)] = v;
        else
            xh[int64_t(m) * kb8 + i] = v;
    };
    if (FRAG && m >= M) {
        for (int i = t; i < kb8; i += 256) put(i, make_uint4(0u, 0u, 0u, 0u));
        return;
    }
    const int ps = hd + 4;
    float4 lo[NR], hi[NR];
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const int i = min(t + 256 * j, kb8 - 1), col = 8 * i, head = col / hd, dim = col % hd;
        float mv[KS], lv[KS];
        float4 ol[KS], oh[KS];
#pragma unroll
        for (int z = 0; z < KS; ++z) {
            if (z < ks) {
                const float* pz = part + ((int64_t(z) * M + m) * n_heads + head) * ps;
                mv[z] = pz[hd];
                lv[z] = pz[hd + 1];
                ol[z] = *reinterpret_cast<const float4*>(pz + dim);
                oh[z] = *reinterpret_cast<const float4*>(pz + dim + 4);
            }
        }
        float Mz = mv[0];
#pragma unroll
        for (int z = 1; z < KS; ++z)
            if (z < ks) Mz = fmaxf(Mz, mv[z]);
        float4 nl = make_float4(0.f, 0.f, 0.f, 0.f), nh = nl;
        float den = 0.f;
#pragma unroll
        for (int z = 0; z < KS; ++z) {
            if (z < ks && mv[z] != -INFINITY) {
                const float w = exp2f(mv[z] - Mz);
                nl = make_float4(fmaf(w, ol[z].x, nl.x), fmaf(w, ol[z].y, nl.y), fmaf(w, ol[z].z, nl.z),
                                 fmaf(w, ol[z].w, nl.w));
                nh = make_float4(fmaf(w, oh[z].x, nh.x), fmaf(w, oh[z].y, nh.y), fmaf(w, oh[z].z, nh.z),
                                 fmaf(w, oh[z].w, nh.w));
                den = fmaf(w, lv[z], den);
            }
        }
        lo[j] = make_float4(nl.x / den, nl.y / den, nl.z / den, nl.w / den);
        hi[j] = make_float4(nh.x / den, nh.y / den, nh.z / den, nh.w / den);
        mx = fmaxf(mx, absmax8(lo[j], hi[j]));
    }
    const float up = row_shift_up(mx, red, xscale + m, t);
#pragma unroll
    for (int j = 0; j < NR; ++j)
        if (t + 256 * j < kb8) put(t + 256 * j, pack_x8(lo[j], hi[j], up));
}
template <bool FRAG, bool SW>
void launch_x_f16r_t(const float* x, const float* u, uint4* xh, float* xscale, int M, int kb8, hipStream_t s) {
    const float4* x4 = reinterpret_cast<const float4*>(x);
    const float4* u4 = reinterpret_cast<const float4*>(u);
    const dim3 g = dim3(unsigned(FRAG ? (M + 31) / 32 * 32 : M)), b = dim3(256);
    if (kb8 <= 256) hipLaunchKernelGGL((k_x_f16r<1, FRAG, SW>), g, b, 0, s, x4, u4, xh, xscale, kb8, M);
    else if (kb8 <= 512) hipLaunchKernelGGL((k_x_f16r<2, FRAG, SW>), g, b, 0, s, x4, u4, xh, xscale, kb8, M);
    else if (kb8 <= 1024) hipLaunchKernelGGL((k_x_f16r<4, FRAG, SW>), g, b, 0, s, x4, u4, xh, xscale, kb8, M);
    else if (kb8 <= 2048) hipLaunchKernelGGL((k_x_f16r<8, FRAG, SW>), g, b, 0, s, x4, u4, xh, xscale, kb8, M);
    else hipLaunchKernelGGL((k_x_f16r<0, FRAG, SW>), g, b, 0, s, x4, u4, xh, xscale, kb8, M);
}
template <bool FRAG>
void launch_x_f16r(const float* x, uint4* xh, float* xscale, int M, int kb8, hipStream_t s) {
    launch_x_f16r_t<FRAG, false>(x, nullptr, xh, xscale, M, kb8, s);
}

// The prompt forward's RMSNorm of a token block straight into the prefill
// GEMM's fp16 operand, one block per row: with `a`, h += a first (per element,
// the updated row written back: the residual add); then the norm with f64
// sums, y = float(x * inv * gamma) in f64 (layers/rmsnorm/cpu.go:70-85, as the
// decoder's k_rmsnorm); then the row's factor and fp16 blocks exactly as
// k_x_f16r<NR, false, false> makes them from y (max|y| in [2^14, 2^15), k
// order [0,2,4,6,1,3,5,7]); with `y`, the f32 rows as well (a and y may be
// the same rows: a block reads its row of a before its first barrier and
// writes y after it). An 8-column block is float4s 2b, 2b + 1, held by lanes
// 2b, 2b + 1; the even lane packs it. FRAG writes the blocks in the
// A-fragment order of GemmArgs::xh, as k_x_f16r<NR, true, false> does: the
// grid covers the M rows padded to 32, and the padding rows get zeros.
// `a` may be the unsummed K split of the GEMM that made it (a_splits
// slices a_stride floats apart, at most 4): the slices are added in split
// order, as k_split_sum adds them, every load issued before the first add.
template <bool FRAG>
__global__ void __launch_bounds__(1024) k_norm_x_f16r(float* __restrict__ h, const float* a, int a_splits,
                                                      int64_t a_stride, const float* __restrict__ gamma, float* y,
                                                      uint4* __restrict__ xh, float* __restrict__ xscale, int dim,
                                                      double eps, int M) {
    __shared__ double part[16];
    __shared__ float redm[16];
    const int m = blockIdx.x, t = threadIdx.x;
    constexpr int R = 4;
    const int n4 = dim / 4, kb8 = dim / 8;
    const int mt = (M + 31) / 32;
    auto put = [&](int b, uint4 v) {
        if constexpr (FRAG)
            xh[(int64_t(b >> 1) * mt + (m >> 5)) * 64 + (m & 31) + 32 * (b & 1)] = v;
        else
            xh[int64_t(m) * kb8 + b] = v;
    };
    if (FRAG && m >= M) {
        for (int b = t; b < kb8; b += 1024) put(b, make_uint4(0u, 0u, 0u, 0u));
        return;
    }
    h += int64_t(m) * dim;
    float4 xv[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = t + 1024 * r;
        xv[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < n4) {
            xv[r] = reinterpret_cast<const float4*>(h)[i];
            if (a) {
                const float4* ap = reinterpret_cast<const float4*>(a + int64_t(m) * dim) + i;
                float4 sv[4];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k < a_splits) sv[k] = ap[(int64_t(k) * a_stride) >> 2];
                float4 av = sv[0];
#pragma unroll
                for (int k = 1; k < 4; ++k)
                    if (k < a_splits) av = make_float4(av.x + sv[k].x, av.y + sv[k].y, av.z + sv[k].z, av.w + sv[k].w);
                xv[r] = make_float4(xv[r].x + av.x, xv[r].y + av.y, xv[r].z + av.z, xv[r].w + av.w);
            }
        }
    }
    double ss = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r)
        ss += double(xv[r].x) * xv[r].x + double(xv[r].y) * xv[r].y + double(xv[r].z) * xv[r].z +
              double(xv[r].w) * xv[r].w;
    ss = wave_total_f64(ss);
    if ((t & 63) == 0) part[t >> 6] = ss;
    __syncthreads();
    double tot = 0.0;
    for (int w = 0; w < 16; ++w) tot += part[w];
    const double inv = 1.0 / sqrt(tot / double(dim) + eps);
    float4 yv[R];
    float mx = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = t + 1024 * r;
        yv[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < n4) {
            if (a) reinterpret_cast<float4*>(h)[i] = xv[r];
            const float4 g = gamma ? reinterpret_cast<const float4*>(gamma)[i] : make_float4(1.f, 1.f, 1.f, 1.f);
            yv[r].x = float(double(xv[r].x) * inv * double(g.x));
            yv[r].y = float(double(xv[r].y) * inv * double(g.y));
            yv[r].z = float(double(xv[r].z) * inv * double(g.z));
            yv[r].w = float(double(xv[r].w) * inv * double(g.w));
            if (y) reinterpret_cast<float4*>(y + int64_t(m) * dim)[i] = yv[r];
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(yv[r].x), fabsf(yv[r].y)), fmaxf(fabsf(yv[r].z), fabsf(yv[r].w))));
        }
    }
    mx = wave_maximum(mx);
    if ((t & 63) == 0) redm[t >> 6] = mx;
    __syncthreads();
    mx = redm[0];
    for (int w = 1; w < 16; ++w) mx = fmaxf(mx, redm[w]);
    int sh = 0;  // the rows are multiplied by 2^sh
    if (mx > 0.f && mx <= 3.4028235e38f) sh = min(126, max(-126, 14 - ilogbf(mx)));
    if (t == 0) xscale[m] = ldexpf(1.0f, -sh);
    const float up = ldexpf(1.0f, sh);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = t + 1024 * r;
        const float4 nb = make_float4(quad_xor1(yv[r].x), quad_xor1(yv[r].y), quad_xor1(yv[r].z), quad_xor1(yv[r].w));
        if (!(t & 1) && i < n4 && i / 2 < kb8) put(i / 2, pack_x8(yv[r], nb, up));
    }
}

// y[i] = sum_k part[k*n + i], k ascending; each thread owns 4 consecutive
// outputs (float4 when n % 4 == 0 and y is 16-byte aligned; the partials
// always are) and issues up to 8 splits' loads before adding them.
__global__ void __launch_bounds__(256) k_split_sum(const float* __restrict__ part, float* __restrict__ y, int64_t n,
                                                  int splits) {
    const int64_t i4 = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i4 * 4 >= n) return;
    if ((n & 3) || (reinterpret_cast<uintptr_t>(y) & 15)) {  // ragged or unaligned: scalar, in the same order
        for (int64_t i = i4 * 4; i < min<int64_t>(n, i4 * 4 + 4); ++i) {
            float s = 0.f;
            for (int k = 0; k < splits; ++k) s += part[int64_t(k) * n + i];
            y[i] = s;
        }
        return;
    }
    const float4* p = reinterpret_cast<const float4*>(part) + i4;
    const int64_t n4 = n >> 2;
    // Splits in order; each group of 8 loads (clamped to the last split, the
    // extra ones masked out of the sum) is issued before any add.
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k = 0; k < splits; k += 8) {
        float4 v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[int64_t(min(k + j, splits - 1)) * n4];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (k + j < splits) {
                s.x += v[j].x;
                s.y += v[j].y;
                s.z += v[j].z;
                s.w += v[j].w;
            }
        }
    }
    reinterpret_cast<float4*>(y)[i4] = s;
}

}  // namespace

// Q4_K at every M; every other row-interleaved format from 9 token rows up
// (up to 8 rows, one batched GEMV launch reads the weights once).
bool gemm_supported(const DevBlob& b, int M) {
    if (b.layout != LAYOUT_RPL) return false;
    if (!b.rpl.wrow) return false;  // the gate/up pair images carry no row factors
    return b.fmt == FMT_Q4_K || M > 8;
}

// Which kernel runs a token block, its tile height (bm tokens), the K split
// (splits of sb_per_split super-blocks) and, for k_gemm_rg, its waves per
// block W and super-blocks per wave `per`:
//   * up to 64 tokens: k_gemm_rg (one block per 64-row group, 8 waves
//     splitting K, one or two 32-token tiles), K split over blocks by the
//     fewest passes of the grid per unit of work (below);
//   * 65 to 128 tokens on at least 200 row groups: k_gemm_rg with four
//     32-token tiles (4 waves, one per SIMD), no K split (4096->14336 M = 128
//     43.5 against 45.7 us; with the split, 14336->4096, 49.3 against 45.0);
//   * 65 to 128 tokens on fewer row groups: k_gemm_rg with two 64-token
//     blocks (8 waves, 2 per SIMD), K split as above (14336->4096 M = 128
//     42.1-42.7 against 42.7-43.4 us on k_gemm_q4k_pw split 14 ways);
//   * otherwise k_gemm_q4k_pw (256-row tiles of 128 or 256 tokens, one block
//     per CU), K split while whole tiles leave CUs idle.
constexpr int kRgMinBlocks = 200;  // row groups on which 128-token k_gemm_rg blocks fill the GPU unsplit
constexpr int64_t kCUs = 256;       // MI355X
int64_t pw_passes(int64_t tiles) { return (tiles + kCUs - 1) / kCUs; }  // of the GPU, one block per CU
GemmPlan gemm_plan(const DevBlob& b, int M) {
    const RplArgs& a = b.rpl;
    GemmPlan p{GEMM_PW, M <= 32 ? 32 : M <= 64 || (M <= 128 && a.rg_count < kRgMinBlocks) ? 64 : 128, 1, a.nsb, 1, 1};
    int want = 1;
    if (M <= 128) {
        // A k_gemm_rg block fills its CU (8 waves of up to 256 registers, or
        // 4 of 512), so the grid runs in ceil(blocks / 256) passes of
        // 1/want of the work each: the split with the fewest passes per unit
        // of work, the smallest of equals (no split sum where a split would
        // only add a pass).
        p.kind = GEMM_RG;
        const int64_t tiles = int64_t(a.rg_count) * ((M + p.bm - 1) / p.bm);
        const int max_split = std::max(1, a.nsb / 8);  // each split >= 8 super-blocks
        double best = 0.0;
        for (int w = 1; w <= max_split; ++w) {
            const double t = double((tiles * w + kCUs - 1) / kCUs) / w;
            if (w == 1 || t < best - 1e-9) {
                best = t;
                want = w;
            }
        }
    } else {
        const int64_t nrow = (a.rows + 255) / 256;
        // 256-token tiles dequantize half as often per product and take 1.82 times a 128-token tile
        // (4096->14336: 131 against 72 us a pass): where that beats the 128-token grid's passes.
        if (1.85 * double(pw_passes(nrow * ((M + 255) / 256))) < double(pw_passes(nrow * ((M + 127) / 128)))) p.bm = 256;
        const int64_t tiles = nrow * ((M + p.bm - 1) / p.bm);
        want = int(std::max<int64_t>(1, 256 / tiles));
        want = std::min(want, std::max(1, a.nsb / 2));  // each split >= 2 super-blocks
    }
    p.sb_per_split = (a.nsb + want - 1) / want;
    p.splits = (a.nsb + p.sb_per_split - 1) / p.sb_per_split;
    if (p.kind == GEMM_RG) {
        p.per = (p.sb_per_split + rg_waves(p.bm / 32) - 1) / rg_waves(p.bm / 32);
        p.W = (p.sb_per_split + p.per - 1) / p.per;
    }
    return p;
}

// Scratch floats: the fp16 copy of X (M*K halves), the M row factors, then
// the split-K partials (each piece 256-byte aligned).
size_t gemm_x_floats(const DevBlob& b, int M) {
    return ((size_t(M) + 31) / 32 * 32 * size_t(b.cols) / 2 + 63) / 64 * 64;  // tokens padded to 32 (A fragments)
}
size_t gemm_scale_floats(int M) { return (size_t(M) + 63) / 64 * 64; }
size_t gemm_scratch_floats(const DevBlob& b, int M) {
    const GemmPlan p = gemm_plan(b, M);
    return gemm_x_floats(b, M) + gemm_scale_floats(M) + (p.splits > 1 ? size_t(p.splits) * size_t(M) * size_t(b.rows) : 0);
}

bool gemm_x_frag(const DevBlob& b, int M) { return gemm_plan(b, M).kind == GEMM_RG; }

int launch_norm_x_f16r(float* h, const float* a, int a_splits, int64_t a_stride, const float* gamma, float* y, void* xh,
                       float* xscale, int M, int dim, double eps, bool frag, void* stream) {
    if (a_splits < 1 || a_splits > 4 || (a_stride & 3)) return int(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (frag)
        hipLaunchKernelGGL(k_norm_x_f16r<true>, dim3(unsigned((M + 31) / 32 * 32)), dim3(1024), 0, s, h, a, a_splits,
                           a_stride, gamma, y, static_cast<uint4*>(xh), xscale, dim, eps, M);
    else
        hipLaunchKernelGGL(k_norm_x_f16r<false>, dim3(unsigned(M)), dim3(1024), 0, s, h, a, a_splits, a_stride, gamma,
                           y, static_cast<uint4*>(xh), xscale, dim, eps, M);
    return 0;
}

int launch_merge_x_f16r(const float* part, int ks, int n_heads, int hd, int M, bool frag, void* xhv, float* xscale,
                        void* stream) {
    const int kb8 = n_heads * hd / 8;
    if (ks < 1 || ks > 8 || hd % 8 || kb8 > 1024) return int(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint4* xh = static_cast<uint4*>(xhv);
    const dim3 g(unsigned(frag ? (M + 31) / 32 * 32 : M)), b(256);
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, g, b, 0, s, part, ks, n_heads, hd, xh, xscale, kb8, M); };
    if (kb8 <= 256) frag ? go(k_merge_x_f16r<1, true>) : go(k_merge_x_f16r<1, false>);
    else if (kb8 <= 512) frag ? go(k_merge_x_f16r<2, true>) : go(k_merge_x_f16r<2, false>);
    else frag ? go(k_merge_x_f16r<4, true>) : go(k_merge_x_f16r<4, false>);
    return 0;
}

void launch_split_sum(const float* part, float* y, int64_t n, int splits, void* stream) {
    hipLaunchKernelGGL(k_split_sum, dim3(unsigned((n / 4 + 1 + 255) / 256)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), part, y, n, splits);
}

void gemm_convert_x(const float* d_x, const float* d_u, int cols, int M, bool frag, void* xhv, float* xscale,
                    void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint4* xh = static_cast<uint4*>(xhv);
    const int kb8 = cols / 8;
    if (frag) {
        if (d_u) launch_x_f16r_t<true, true>(d_x, d_u, xh, xscale, M, kb8, s);
        else launch_x_f16r_t<true, false>(d_x, nullptr, xh, xscale, M, kb8, s);
    } else {
        if (d_u) launch_x_f16r_t<false, true>(d_x, d_u, xh, xscale, M, kb8, s);
        else launch_x_f16r_t<false, false>(d_x, nullptr, xh, xscale, M, kb8, s);
    }
}

namespace {
struct PartOf {  // the part of gemm_tiles.hip that has the kernels of a format's builder
    bool tall;    // 256-token tiles
    int& part;
    template <class GP>
    void run() const {
        part = gemm_part<GP>(tall);
    }
};
}  // namespace

int launch_gemm_xh(const DevBlob& b, const void* xh, const float* xscale, float* d_y, int M, void* stream,
                   float* d_part, int* d_splits) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (!gemm_supported(b, M)) return int(hipErrorInvalidValue);
    const GemmPlan p = gemm_plan(b, M);
    const int bm = p.bm, splits = p.splits;
    if (splits > 1 && !d_part) return int(hipErrorInvalidValue);
    GemmArgs ga;
    ga.w = b.rpl;
    ga.xh = static_cast<const uint4*>(xh);
    ga.xscale = xscale;
    ga.y = splits > 1 ? d_part : d_y;
    ga.M = M;
    ga.K = int(b.cols);
    ga.sb_per_split = p.sb_per_split;
    const dim3 grid(unsigned(p.kind == GEMM_RG ? b.rpl.rg_count : (b.rows + 255) / 256), unsigned((M + bm - 1) / bm),
                    unsigned(splits));
    int part = 0;
    int e = with_builder(b, PartOf{bm == 256, part});
    if (e) return e;
    using Tiles = int (*)(const DevBlob&, const GemmPlan&, dim3, hipStream_t, const GemmArgs&);
    constexpr Tiles tiles[kGemmParts] = {launch_gemm_tiles<0>, launch_gemm_tiles<1>, launch_gemm_tiles<2>,
                                         launch_gemm_tiles<3>, launch_gemm_tiles<4>, launch_gemm_tiles<5>,
                                         launch_gemm_tiles<6>, launch_gemm_tiles<7>};
    e = tiles[part](b, p, grid, s, ga);
    if (e) return e;
    if (d_splits) *d_splits = splits;
    if (splits > 1 && !d_splits) launch_split_sum(d_part, d_y, int64_t(M) * b.rows, splits, s);
    return int(hipGetLastError());
}

int launch_gemm(const DevBlob& b, const float* d_x, float* d_y, int M, void* stream, float* d_scratch) {
    if (!gemm_supported(b, M) || !d_scratch) return int(hipErrorInvalidValue);
    uint4* xh = reinterpret_cast<uint4*>(d_scratch);
    float* xscale = d_scratch + gemm_x_floats(b, M);
    float* part = xscale + gemm_scale_floats(M);
    gemm_convert_x(d_x, nullptr, int(b.cols), M, gemm_x_frag(b, M), xh, xscale, stream);
    return launch_gemm_xh(b, xh, xscale, d_y, M, stream, part);
}

}  // namespace wv
