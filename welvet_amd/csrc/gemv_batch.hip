// gemv_batch.hip — the batched forward Y[b] = W X[b] (b = 2.. rows) at f32
// precision on the row-interleaved layouts: Dense's forward of a batch
// (forwardSIMDBlockFused, layers/dense/simd_block.go:17-39) through
// wv_matvec* and wv_dense_forward*, whose bar is the 1e-5 of the one-row GEMV
// and not the 2e-3 of the fp16 prefill GEMM.
//
// The one-row kernel (gemv_rpl.hip) dequantizes per row of the batch, so its
// time grows with the batch while HBM idles. Here a block decodes each weight
// once for 8 or 16 batch rows and takes the products on the matrix cores,
// exactly enough for f32:
//   * the codes are the B operand of v_mfma_f32_32x32x16_f16 as they are,
//     integers exact in fp16 (GP::codes); a 16-column step is one group of
//     the 16-column formats, so scales stay out of the products;
//   * each f32 x is two fp16 halves, x * 2^s = hi + 2^-12 lo, hi the nearest
//     fp16 and lo the nearest to 2^12 times the remainder (exact in f32), with
//     2^s taking the row's largest |x| of the super-block into [2^14, 2^15):
//     the pair is within 2^-23 of x (f32's own rounding is 2^-24) down to
//     2^-28 of the largest and within 2^-51 of the largest below, where
//     the one-row kernels' fixed point holds 2^-23 of a 32-column chunk's
//     largest. Without the 2^12, lo's smallest step left 2^-39, and a dead
//     channel of 1e8 beside N(0, 1) cost Q4_1 2.9e-5. hi and lo are different
//     rows of the A operand, so one product gives both sums of 8 or 16 batch rows.
//     The 16-column sums of x that meet the k-quants' byte mins are such pairs
//     of a 32nd of the sum, within 2^-46 of the largest x;
//   * D holds exact products summed in f32; the group's scale meets it in f32
//     FMAs on the VALU, 2^-s once per super-block.
// Measured (Q4_K, us a call, one-row kernel before): 4096->14336 13.4 / 14.2 /
// 19.9 at 2 / 8 / 16 rows against 13.8 / 37 / 72; 14336->4096 8 rows 16.7
// against 65; Q8_0 4096->4096 32 rows 14.6 against 89. 2-norm error against f64, 8 rows: 5.5e-7 through gate, up and down
// against 1.4e-6; Q8_0 1.1e-7 against 3.2e-7. What bounds it: at 8 rows the
// weights would stream in 8 us; a wave's VALU work (about 630 instructions a
// super-block for the operands and sums, 450 for converting 8 rows of x) and
// its load latencies at two waves per SIMD overlap only in part. 16 waves of
// 128 registers spilled (24 us), and a form whose 8 waves share one
// converted x, a chunk each, ran 19 us: its per-chunk metadata loads fill the
// L1 (16 lines for 256 bytes).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "rpl_operands.h"
#include "wave_ops.h"
#include "wv_internal.h"

namespace wv {
namespace {

struct GemvBArgs {
    RplArgs w;  // w.partial, w.ksplit: the K split, as k_gemv_rpl's
    const float* x;
    float* y;
    int batch;
    int sb_per_split, per;  // super-blocks per K split and per wave
};

// Formats whose mins are bytes (the k-quants') take the min term once per
// super-block on the matrix cores; the others with an offset (kMin) per scale
// group on the VALU.
template <class GP, class = void>
struct MinBytes : std::false_type {};
template <class GP>
struct MinBytes<GP, std::void_t<decltype(GP::kMinBytes)>> : std::true_type {};

// LDS of one wave, in dwords: the A operand of a super-block (32 rows (k16
// step, half) of 16 NQ slots of 16 bytes, 8 NQ batch rows' hi and then their
// lo, each row padded by 16 bytes so that the staging stores of 16 rows spread
// over the banks), the group sums of x as the A operand of the min product
// (two such rows) or as floats, and 2^-s.
template <int NQ>
struct GemvBLds {
    static constexpr int kRow = 16 * NQ * 4 + 4, kSum = 32 * kRow;
    static constexpr int kInv = kSum + 2 * kRow, kWave = kInv + 8 * NQ;
    static_assert(16 * 8 * NQ <= 2 * kRow && kWave % 4 == 0, "group sums");
};
constexpr int kBWaves = 8;  // per block at most: two of 256 registers on each SIMD

constexpr uint32_t kInfBits = 0x7F800000u;
constexpr uint32_t kLoBits = 12;  // lo halves are held at 2^12 times their place
constexpr float kLoScale = float(1u << kLoBits);
__device__ __forceinline__ uint32_t abs_bits(float f) { return __float_as_uint(f) & 0x7FFFFFFFu; }
__device__ __forceinline__ uint32_t max4_bits(float4 v) {
    const uint32_t a = max(abs_bits(v.x), abs_bits(v.y)), b = max(abs_bits(v.z), abs_bits(v.w));
    return max(a, b);
}
__device__ __forceinline__ float finite_or_0(float f) { return abs_bits(f) < kInfBits ? f : 0.f; }
__device__ __forceinline__ float4 finite_or_0(float4 v) {
    return make_float4(finite_or_0(v.x), finite_or_0(v.y), finite_or_0(v.z), finite_or_0(v.w));
}
// The largest of four values per lane over the wave, one per batch row: two
// lane swaps leave row i's in the 16-lane row i, where four DPP steps finish.
__device__ __forceinline__ void wave_max4(const uint32_t (&m)[4], uint32_t (&out)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(m[0], m[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(m[1], m[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(max(uint32_t(a[0]), uint32_t(a[1])),
                                                    max(uint32_t(b[0]), uint32_t(b[1])), false, false);
    uint32_t v = max(uint32_t(c[0]), uint32_t(c[1]));
    v = max(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x128, 0xf, 0xf, false)));
    v = max(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x124, 0xf, 0xf, false)));
    v = max(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x122, 0xf, 0xf, false)));
    v = max(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x121, 0xf, 0xf, false)));
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = uint32_t(__builtin_amdgcn_readlane(int(v), 16 * i));
}
// The exponent fields of the four rows' 2^s, which takes their largest finite
// |x| into [2^14, 2^15); whether an x of theirs is not finite.
__device__ __forceinline__ bool scale_fields(const float4 (&v)[4], uint32_t (&f)[4]) {
    uint32_t m[4], w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = max4_bits(v[i]);
    wave_max4(m, w);
    const bool odd = max(max(w[0], w[1]), max(w[2], w[3])) >= kInfBits;
    if (odd) {
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = max4_bits(finite_or_0(v[i]));
        wave_max4(m, w);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = min(254u - kLoBits, 268u - (w[i] >> 23));
    return odd;
}
// The fp16 nearest 2^-12 x of a pair, and the remainders x - 2^12 h, exact (|x|
// <= 2^27) until they too are rounded to fp16 (at most 2^15): an instruction a
// half, 3 an element with the scaling. From float code the compiler takes 4.5
// (the remainder's product, a conversion): 8 rows of Q4_K 4096->14336 14.9 us so
// against 14.2, 16 rows of Q8_0 14336->4096 24.1 against 23.3.
__device__ __forceinline__ uint32_t hi_pair(float a, float b) {
    uint32_t h;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(h) : "v"(a), "s"(1.0f / kLoScale));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(h) : "v"(b), "s"(1.0f / kLoScale));
    return h;
}
__device__ __forceinline__ uint32_t lo_pair(uint32_t h, float a, float b) {
    uint32_t l;
    asm("v_fma_mixlo_f16 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(l) : "v"(h), "s"(-kLoScale), "v"(a));
    asm("v_fma_mixhi_f16 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(l) : "v"(h), "s"(-kLoScale), "v"(b));
    return l;
}
__device__ __forceinline__ float rest(float x, _Float16 h) { return fmaf(float(h), -kLoScale, x); }
// lo_pair with 0 for a remainder that is not finite (inf - inf)
__device__ __forceinline__ uint32_t lo_pair_finite(uint32_t hb, float a, float b) {
    const half2v h = __builtin_bit_cast(half2v, hb);
    return pack_h2(finite_or_0(rest(a, h.x)), finite_or_0(rest(b, h.y)));
}
// The sum of a product's hi and lo rows.
__device__ __forceinline__ float hi_lo(float hi, float lo) { return fmaf(lo, 1.0f / kLoScale, hi); }

// One block: 64 rows x 8 NQ batch rows x one K split, its W waves `per`
// consecutive super-blocks each. Per super-block a wave converts its x into
// its own LDS slice (nobody else reads it: no block barrier in the loop), four
// chunks of codes in flight, then runs the 8 chunks. Row i of a product's D is
// batch row i % (8 NQ), from its hi for i < 8 NQ, else from its lo; D row
// 8(r / 4) + 4(l / 32) + r % 4 is register r of lane l, so registers r and
// 4 NQ + r add up to batch row 8(r / 4) + 4(l / 32) + r % 4 of weight row 32T
// + l % 32. The waves' sums meet in LDS in wave order.
template <class GP, int NQ>
__global__ void __launch_bounds__(64 * kBWaves) k_gemv_b(GemvBArgs ga) {
    using L = GemvBLds<NQ>;
    constexpr int NT = 8 * NQ, NR = 4 * NQ, D = 4;  // D chunks of codes in flight
    constexpr int GW = GP::kTwo ? 16 : 32;  // columns per scale
    constexpr int NG = 32 / GW;             // scales per chunk
    constexpr bool kMB = MinBytes<GP>::value, kVM = GP::kMin && !kMB;
    extern __shared__ float4 smb4[];
    float* sm = reinterpret_cast<float*>(smb4);
    const RplArgs& a = ga.w;
    const int t = threadIdx.x, lane = t & 63, W = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int g = blockIdx.x, b0 = blockIdx.y * NT, ks = blockIdx.z;
    const int nt = min(NT, ga.batch - b0);
    const int sb0 = ks * ga.sb_per_split + wave * ga.per;
    const int sb1 = min(min(a.nsb, (ks + 1) * ga.sb_per_split), sb0 + ga.per);
    const int64_t cols = int64_t(a.nsb) * 256;
    float* xs = sm + wave * L::kWave;

    float acc[2][NR];
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[T][r] = 0.f;

    if (sb0 < sb1) {
        const float* xb = ga.x + int64_t(b0) * cols + 4 * lane;
        auto load_x = [&](int sb, int q, float4 (&v)[4]) {  // rows past the batch repeat its last one
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] = *reinterpret_cast<const float4*>(xb + int64_t(min(q + i, nt - 1)) * cols + int64_t(sb) * 256);
        };
        auto load_c = [&](int sb, int j) {
            return GP::load_codes(a, rpl_chunk(a, int64_t(g) * a.nsb + sb, j), lane);
        };
        // x first: vector loads retire in issue order, and the conversion waits for it alone
        float4 xv[NT / 4][4];
#pragma unroll
        for (int q = 0; q < NT / 4; ++q)
            if (4 * q < nt) load_x(sb0, 4 * q, xv[q]);
        typename GP::Meta mt = GP::load_meta(a, int64_t(g) * a.nsb + sb0, lane);
        typename GP::Codes ring[D];
#pragma unroll
        for (int j = 0; j < D; ++j) ring[j] = load_c(sb0, j);
        const int arow = (lane & (2 * NT - 1)) * 4 + (lane >> 5) * L::kRow;  // this lane's A slot in a k16 step
        // lane l holds columns 4l..4l+3 of the super-block: k16 step l / 4, half (l / 2) % 2, 8-byte part l % 2
        float* xw = xs + (lane >> 1) * L::kRow + (lane & 1) * 2;
        _Float16* sw = reinterpret_cast<_Float16*>(xs + L::kSum + (lane >> 5) * L::kRow) + ((lane >> 2) & 7);
        for (int sb = sb0; sb < sb1; ++sb) {
            // Four batch rows at a time (rows past the batch repeat its last one and go nowhere).
#pragma unroll
            for (int q = 0; q < NT; q += 4) {
                if (q >= nt) break;
                float4 (&v)[4] = xv[q / 4];
                uint32_t f[4];
                const bool odd = scale_fields(v, f);
                float sum[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float up = __uint_as_float((f[i] + kLoBits) << 23);
                    v[i] = make_float4(v[i].x * up, v[i].y * up, v[i].z * up, v[i].w * up);
                    if constexpr (GP::kMin) sum[i] = (v[i].x + v[i].y) + (v[i].z + v[i].w);
                }
                uint2 h[4], d[4];  // columns 0 | 2 and 1 | 3
                if (!odd) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        h[i] = make_uint2(hi_pair(v[i].x, v[i].z), hi_pair(v[i].y, v[i].w));
                        d[i] = make_uint2(lo_pair(h[i].x, v[i].x, v[i].z), lo_pair(h[i].y, v[i].y, v[i].w));
                    }
                } else {
                    // A non-finite x takes part as itself, in the code products and in the group sums, and
                    // leaves no output of its row finite. With f32 mins, whose group's products and sum may
                    // be infinities of opposite signs, it does so through the sum alone, as in the one-row kernels.
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float4 w = kVM ? finite_or_0(v[i]) : v[i];
                        h[i] = make_uint2(hi_pair(w.x, w.z), hi_pair(w.y, w.w));
                        d[i] = make_uint2(lo_pair_finite(h[i].x, w.x, w.z), lo_pair_finite(h[i].y, w.y, w.w));
                    }
                }
                if constexpr (GP::kMin) {  // the group sums of x, in every lane of a group; four rows hide a DPP's wait
#pragma unroll
                    for (int i = 0; i < 4; ++i) sum[i] += quad_xor1(sum[i]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) sum[i] += quad_xor2(sum[i]);
                    if constexpr (GW == 32) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) sum[i] += half_mirror(sum[i]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    *reinterpret_cast<uint2*>(xw + (q + i) * 4) = h[i];
                    *reinterpret_cast<uint2*>(xw + (NT + q + i) * 4) = d[i];
                    xs[L::kInv + q + i] = __uint_as_float((254u - f[i]) << 23);
                    if constexpr (GP::kMin) {  // the lanes of a group store the same sum
                        float S = sum[i];
                        if constexpr (kMB) {
                            S *= 0.03125f;  // at most 2^26
                            const _Float16 sh = _Float16(S * (1.0f / kLoScale));
                            sw[(q + i) * 8] = sh;
                            sw[(NT + q + i) * 8] = _Float16(odd ? finite_or_0(rest(S, sh)) : rest(S, sh));
                        } else {
                            xs[L::kSum + (lane / (GW / 4)) * NT + q + i] = S * (1.0f / kLoScale);
                        }
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int nx = min(sb + 1, sb1 - 1);
            float s[2][NR];
#pragma unroll
            for (int T = 0; T < 2; ++T)
#pragma unroll
                for (int r = 0; r < NR; ++r) s[T][r] = 0.f;
            uint32_t mb[8];
            half8 bf[2][2];
            float sc[2][2], mn[2][2];
            auto build = [&](int j) {
                const typename GP::Ch ch = GP::chunk(ring[j % D], mt, j);
                GP::codes(ch, lane, bf);
                GP::scales(ch, sc, mn);
                if constexpr (kMB) mb[j] = GP::min_codes(ch);
            };
            build(0);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                ring[j % D] = j + D < 8 ? load_c(sb, j + D) : load_c(nx, j + D - 8);
                half8 af[2];
#pragma unroll
                for (int kk = 0; kk < 2; ++kk)
                    af[kk] = *reinterpret_cast<const half8*>(xs + (2 * j + kk) * 2 * L::kRow + arow);
                const f32x16 z = {};
                f32x16 d[2][NG];  // the products of all columns of a scale group
#pragma unroll
                for (int T = 0; T < 2; ++T) {
                    d[T][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[0], bf[T][0], z, 0, 0, 0);
                    d[T][NG - 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[1], bf[T][1], NG == 2 ? z : d[T][0], 0, 0, 0);
                }
                float cs[2][2], ms[2][2];
#pragma unroll
                for (int T = 0; T < 2; ++T)
#pragma unroll
                    for (int kk = 0; kk < NG; ++kk) {
                        cs[T][kk] = sc[T][kk];
                        if constexpr (kVM) ms[T][kk] = mn[T][kk];
                    }
                __builtin_amdgcn_sched_barrier(0);
                if (j < 7) build(j + 1);  // beside the products
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int T = 0; T < 2; ++T)
#pragma unroll
                    for (int kk = 0; kk < NG; ++kk)
#pragma unroll
                        for (int r = 0; r < NR; ++r) s[T][r] = fmaf(hi_lo(d[T][kk][r], d[T][kk][NR + r]), cs[T][kk], s[T][r]);
                if constexpr (kVM) {
#pragma unroll
                    for (int kk = 0; kk < NG; ++kk)
#pragma unroll
                        for (int o = 0; o < NQ; ++o) {
                            const float4 S = *reinterpret_cast<const float4*>(
                                xs + L::kSum + (j * NG + kk) * NT + 8 * o + 4 * (lane >> 5));
#pragma unroll
                            for (int T = 0; T < 2; ++T) {
                                s[T][4 * o] = fmaf(ms[T][kk], S.x, s[T][4 * o]);
                                s[T][4 * o + 1] = fmaf(ms[T][kk], S.y, s[T][4 * o + 1]);
                                s[T][4 * o + 2] = fmaf(ms[T][kk], S.z, s[T][4 * o + 2]);
                                s[T][4 * o + 3] = fmaf(ms[T][kk], S.w, s[T][4 * o + 3]);
                            }
                        }
                }
                // the chunk's sums are done here: left free, the compiler keeps every chunk's products
                // and spills them
#pragma unroll
                for (int T = 0; T < 2; ++T)
#pragma unroll
                    for (int r = 0; r < NR; ++r) asm volatile("" : "+v"(s[T][r]));
            }
            if constexpr (kMB) {
                // B: groups 0-7 in lanes 0-31 and 8-15 in lanes 32-63 of a 32-row tile's rows
                uint32_t bm[2][4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const auto r = __builtin_amdgcn_permlane32_swap(mb[k], mb[k + 4], false, false);
                    bm[0][k] = r[0];
                    bm[1][k] = r[1];
                }
                float dm[2];
                GP::min_scale(mt, dm);
                const half8 sa = *reinterpret_cast<const half8*>(xs + L::kSum + arow);
                const f32x16 z = {};
#pragma unroll
                for (int T = 0; T < 2; ++T) {
                    const half8 b8 = __builtin_bit_cast(half8, make_uint4(bm[T][0], bm[T][1], bm[T][2], bm[T][3]));
                    const f32x16 d = __builtin_amdgcn_mfma_f32_32x32x16_f16(sa, b8, z, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < NR; ++r) s[T][r] = fmaf(hi_lo(d[r], d[NR + r]), dm[T], s[T][r]);
                }
            }
#pragma unroll
            for (int o = 0; o < NQ; ++o) {
                const float4 I = *reinterpret_cast<const float4*>(xs + L::kInv + 8 * o + 4 * (lane >> 5));
#pragma unroll
                for (int T = 0; T < 2; ++T) {
                    acc[T][4 * o] = fmaf(s[T][4 * o], I.x, acc[T][4 * o]);
                    acc[T][4 * o + 1] = fmaf(s[T][4 * o + 1], I.y, acc[T][4 * o + 1]);
                    acc[T][4 * o + 2] = fmaf(s[T][4 * o + 2], I.z, acc[T][4 * o + 2]);
                    acc[T][4 * o + 3] = fmaf(s[T][4 * o + 3], I.w, acc[T][4 * o + 3]);
                }
            }
            if (sb + 1 < sb1) {
#pragma unroll
                for (int q = 0; q < NT / 4; ++q)
                    if (4 * q < nt) load_x(nx, 4 * q, xv[q]);
                mt = GP::load_meta(a, int64_t(g) * a.nsb + nx, lane);
            }
            // the next super-block's staging stores follow these reads
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }

    __syncthreads();  // every wave is done with its slice
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
        for (int r = 0; r < NR; ++r) sm[((wave * 2 + T) * NR + r) * 64 + lane] = acc[T][r];
    __syncthreads();
    const int64_t rows_pad = int64_t(a.rg_count) * 64;
    for (int v = t; v < NT * 64; v += 64 * W) {  // v = (batch row, weight row)
        const int i = v >> 6, n = v & 63, T = n >> 5;
        const int r = 4 * (i >> 3) + (i & 3), l = (n & 31) + 32 * ((i >> 2) & 1);
        float sum = 0.f;
        for (int w = 0; w < W; ++w) sum += sm[((w * 2 + T) * NR + r) * 64 + l];
        if (i >= nt) continue;
        const int row = g * 64 + n;
        if (a.ksplit > 1)
            a.partial[(int64_t(b0 + i) * a.ksplit + ks) * rows_pad + row] = sum;
        else if (row < a.rows)
            ga.y[int64_t(b0 + i) * a.rows + row] = sum;
    }
}

// NQ octets of batch rows per block, W waves of `per` super-blocks each, K
// split over blocks (splits of sb_per_split super-blocks).
struct GemvBPlan {
    int nq, W, per, splits, sb_per_split;
};
constexpr int64_t kBCUs = 256;  // MI355X
GemvBPlan gemv_b_plan(const DevBlob& b, int batch) {
    const RplArgs& a = b.rpl;
    GemvBPlan p;
    p.nq = batch <= 8 ? 1 : 2;
    const int64_t blocks = int64_t(a.rg_count) * ((batch + 8 * p.nq - 1) / (8 * p.nq));
    // K splits while whole blocks leave CUs idle, at least 4 super-blocks each:
    // at most 256 / blocks of them, so at most 2^18 floats of partials.
    const int want = int(std::max<int64_t>(1, std::min<int64_t>(kBCUs / blocks, a.nsb / 4)));
    p.sb_per_split = (a.nsb + want - 1) / want;
    p.splits = (a.nsb + p.sb_per_split - 1) / p.sb_per_split;
    p.per = (p.sb_per_split + kBWaves - 1) / kBWaves;
    p.W = (p.sb_per_split + p.per - 1) / p.per;
    return p;
}

template <int NQ>
struct GemvBGo {
    dim3 grid;
    const GemvBPlan& p;
    hipStream_t s;
    const GemvBArgs& ga;
    template <class GP>
    void run() const {
        if constexpr (GP::kExact) {
            const size_t lds = sizeof(float) * size_t(p.W) * std::max(GemvBLds<NQ>::kWave, 2 * 4 * NQ * 64);
            hipLaunchKernelGGL((k_gemv_b<GP, NQ>), grid, dim3(unsigned(64 * p.W)), lds, s, ga);
        }
    }
};

}  // namespace

// A launch takes 9-13 us however few weights it has (a wave's chain of x,
// conversion and chunks, and the K split's second launch on few rows), where
// the one-row kernels take 4-5 us plus 0.07 us (Q8_0 0.12 or more) per million
// weights and batch row. The lines are where both sides met on a grid of 9
// shapes from 1024x4096 to 14336x4096 and 2 to 32 rows, weights x rows: Q4_K
// 9.3 against 10.0 us here at 67 M, 13.2 against 12.6 at 94 M, 14.8 against
// 11.4 at 126 M; Q6_K and Q4_0 alike; Q8_0 8 rows and fewer 13.3 against 12.1
// at 44 M, 15.4 against 10.0 at 67 M, more rows 10.9 against 11.8 at 67 M, 14.1
// against 10.4 at 94 M. IQ4_NL's float grid is not exact in fp16.
// Two and three rows leave most of an octet's work unused, so there the two
// plans' times are compared (Q8_0 apart, which gains everywhere): a pass of the
// batched kernel over the GPU takes 5 us and 6 for each super-block of a wave,
// a K split 2 more, the one-row kernel what gemv_b_row_us says. Q4_K 2 rows:
// 20555x2560, two passes, 22.0 us against the one-row kernel's 12.7;
// 44096x1536 22.8 against 15.7; 4096x14336 16.3 against 18.2. Of 705 calls
// (19 formats, 37 shapes) 11 run over 2.5 % slower than on the one-row kernel, to
// 10 %, and 40 would gain as much here; with the lines above alone 205 ran
// slower, to 43 %.
static double gemv_b_row_us(int fmt) {  // us per million weights and row
    switch (fmt) {
    case FMT_Q2_K: return 0.105;
    case FMT_Q6_K: case FMT_Q4_0: case FMT_Q5_0: return 0.165;
    case FMT_IQ2_XS: case FMT_IQ3_S: case FMT_IQ4_XS: case FMT_TERNARY: return 0.17;
    case FMT_Q4_1: case FMT_Q5_1: return 0.185;
    default: return 0.13;
    }
}
bool gemv_b_supported(const DevBlob& b, int batch) {
    if (batch < 2 || b.layout != LAYOUT_RPL || b.fmt == FMT_IQ4_NL) return false;
    const double work = double(batch) * double(b.rows) * double(b.cols);
    if (work < (b.fmt != FMT_Q8_0 ? 105e6 : batch <= 8 ? 60e6 : 90e6)) return false;
    if (batch > 3 || b.fmt == FMT_Q8_0) return true;
    const GemvBPlan p = gemv_b_plan(b, batch);
    // blocks of up to 4 waves run two to a CU
    const int64_t blocks = int64_t(b.rpl.rg_count) * p.splits, fit = p.W <= 4 ? 2 * kBCUs : kBCUs;
    const double passes = double((blocks + fit - 1) / fit);
    return 6.0 + gemv_b_row_us(b.fmt) * work * 1e-6 >= passes * (5.0 + 6.0 * p.per) + (p.splits > 1 ? 2.0 : 0.0);
}

size_t gemv_b_scratch_floats(const DevBlob& b, int batch) {
    const GemvBPlan p = gemv_b_plan(b, batch);
    return p.splits > 1 ? size_t(batch) * size_t(p.splits) * size_t(b.rpl.rg_count) * 64 : 0;
}

int launch_gemv_b(const DevBlob& b, const float* d_x, float* d_y, int batch, void* stream, float* d_scratch) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    constexpr int kMaxRows = 65535 * 8;  // the grid's y limit
    // One plan for every part of a batch past the limit, the one that the
    // scratch was sized for: a short last part planned by itself would split K.
    const GemvBPlan p = gemv_b_plan(b, batch);
    if (p.splits > 1 && !d_scratch) return int(hipErrorInvalidValue);
    for (int r0 = 0; r0 < batch; r0 += kMaxRows) {
        const int nb = std::min(kMaxRows, batch - r0);
        GemvBArgs ga;
        ga.w = b.rpl;
        ga.w.mode = RPL_STORE;
        ga.w.aux = nullptr;
        ga.w.ss_out = nullptr;
        ga.w.partial = d_scratch;
        ga.w.ksplit = p.splits;
        ga.x = d_x + int64_t(r0) * b.cols;
        ga.y = d_y + int64_t(r0) * b.rows;
        ga.batch = nb;
        ga.sb_per_split = p.sb_per_split;
        ga.per = p.per;
        const dim3 grid(unsigned(b.rpl.rg_count), unsigned((nb + 8 * p.nq - 1) / (8 * p.nq)), unsigned(p.splits));
        const int e = p.nq == 1 ? with_builder(b, GemvBGo<1>{grid, p, s, ga}) : with_builder(b, GemvBGo<2>{grid, p, s, ga});
        if (e) return e;
        if (p.splits > 1) launch_rpl_ksum(ga.w, ga.y, nb, s);
    }
    return int(hipGetLastError());
}

}  // namespace wv
