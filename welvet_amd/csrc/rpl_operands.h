// rpl_operands.h — the row-interleaved code planes as MFMA B operands.
//
// Loaders and per-format builders shared by the batched kernels of the
// row-interleaved layouts: the prefill GEMM (gemm_rpl.hip), whose operands are
// dequantized fp16 weights, and the f32-precision batched forward
// (gemv_batch.hip), whose operands are the codes themselves.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "wave_ops.h"
#include "wv_internal.h"

namespace wv {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));


__device__ __forceinline__ uint4 ld_nt(const uint4* p) {
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
    const half2v h = {_Float16(a), _Float16(b)};
    return __builtin_bit_cast(uint32_t, h);
}

// 8 weights from two spread words (byte b of `se` / `so` = the code of
// column 2b / 2b + 1 of an 8-column run) -> 4 half2 w = fma(q, sc, mn) in
// fp16, in k order [0,2,4,6,1,3,5,7].
// Codes of up to 4 bits convert with v_cvt_scalef32_pk_f16_fp8: a byte q <
// 16 read as fp8 e4m3 is q * 2^-9 exactly (exponent fields 0 and 1 share the
// step 2^-9), and the instruction applies the exponent of its f32 scale, so
// scale 512 gives q as fp16 for two bytes in one instruction. Wider codes
// (up to 5 bits) take the exponent-byte form: 0x64 | q is 1024 + q in fp16.
template <int FB>
__device__ __forceinline__ uint4 dequant8s(uint32_t se, uint32_t so, half2v sc, half2v mn) {
    half2v q[4];
    if constexpr (FB <= 4) {
        q[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(se, 512.0f, false);
        q[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(se, 512.0f, true);
        q[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(so, 512.0f, false);
        q[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(so, 512.0f, true);
    } else {
        const half2v k1024 = {_Float16(1024.0f), _Float16(1024.0f)};
        const uint32_t e = 0x64646464u;
        q[0] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(e, se, 0x04010400u)) - k1024;
        q[1] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(e, se, 0x04030402u)) - k1024;
        q[2] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(e, so, 0x04010400u)) - k1024;
        q[3] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(e, so, 0x04030402u)) - k1024;
    }
    uint32_t p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = __builtin_bit_cast(uint32_t, q[i] * sc + mn);
    return make_uint4(p[0], p[1], p[2], p[3]);
}

// The exact form for k_gemv_b: 8 codes minus MID2 / 2 as fp16 integers (or
// halves), unscaled, in k order [0,2,1,3,4,6,5,7].
template <int FB, int MID2>
__device__ __forceinline__ half8 codes8(uint32_t se, uint32_t so) {
    half2v q[4];
    if constexpr (FB <= 4) {
        q[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(se, 512.0f, false);
        q[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(so, 512.0f, false);
        q[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(se, 512.0f, true);
        q[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(so, 512.0f, true);
        if constexpr (MID2 != 0) {
            const half2v mid = {_Float16(0.5f * MID2), _Float16(0.5f * MID2)};
#pragma unroll
            for (int i = 0; i < 4; ++i) q[i] -= mid;
        }
    } else {
        static_assert(MID2 % 2 == 0, "1024 + mid is an fp16 integer");
        const half2v mid = {_Float16(1024.0f + 0.5f * MID2), _Float16(1024.0f + 0.5f * MID2)};
        const uint32_t e = 0x64646464u;
        q[0] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(e, se, 0x04010400u)) - mid;
        q[1] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(e, so, 0x04010400u)) - mid;
        q[2] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(e, se, 0x04030402u)) - mid;
        q[3] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(e, so, 0x04030402u)) - mid;
    }
    return __builtin_bit_cast(half8, make_uint4(__builtin_bit_cast(uint32_t, q[0]), __builtin_bit_cast(uint32_t, q[1]),
                                                __builtin_bit_cast(uint32_t, q[2]), __builtin_bit_cast(uint32_t, q[3])));
}
// codes8 of both 32-row tiles and k16 steps.
template <int FB, int MID2>
__device__ __forceinline__ void codes_all(const uint32_t (&se)[2][2], const uint32_t (&so)[2][2], half8 (&bf)[2][2]) {
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) bf[T][kk] = codes8<FB, MID2>(se[T][kk], so[T][kk]);
}
// A per-row float of the lane's own row -> out[T], the value of row 32T + lane % 32.
__device__ __forceinline__ void tile_rows(float v, float& t0, float& t1) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    t0 = __uint_as_float(uint32_t(r[0]));
    t1 = __uint_as_float(uint32_t(r[1]));
}

// Code planes of one 32-column chunk of a k-quant row (lane = row) and, after
// the lane swaps, the spread words of the MFMA B operands: for 32-row tile T
// and k16 step kk, lanes 0-31 take columns 16kk + 0..7 of rows 32T + lane and
// lanes 32-63 columns 16kk + 8..15 of the same rows. FB = code bits (2, 3, 4,
// 5); the planes are those of the forward kernels (Q4_K nibbles; Q5_K fifth
// bits; Q2_K / Q3_K two-bit plane and third bits).
template <int FB>
struct GemmCodes {
    struct C { uint4 c; uint32_t h; };
    static __device__ __forceinline__ C load(const RplArgs& a, int64_t ci, int lane) {
        C r;
        if constexpr (FB >= 4) {
            r.c = ld_nt(reinterpret_cast<const uint4*>(a.codes) + ci * 64 + lane);
        } else {
            const uint2 v = reinterpret_cast<const uint2*>(a.codes)[ci * 64 + lane];
            r.c = make_uint4(v.x, v.y, 0u, 0u);
        }
        r.h = (FB == 5 || FB == 3) ? reinterpret_cast<const uint32_t*>(a.hi)[ci * 64 + lane] : 0u;
        return r;
    }
    // se/so[T][kk]: even / odd columns of the lane's 8-column run
    static __device__ __forceinline__ void spread(const C& c, int lane, uint32_t (&se)[2][2], uint32_t (&so)[2][2]) {
        const int up = lane >> 5;
        if constexpr (FB >= 4) {
            const auto k0 = __builtin_amdgcn_permlane32_swap(c.c.x, c.c.y, false, false);  // columns 0-15
            const auto k1 = __builtin_amdgcn_permlane32_swap(c.c.z, c.c.w, false, false);  // columns 16-31
#pragma unroll
            for (int T = 0; T < 2; ++T) {
                se[T][0] = k0[T] & 0x0F0F0F0Fu;
                so[T][0] = (k0[T] >> 4) & 0x0F0F0F0Fu;
                se[T][1] = k1[T] & 0x0F0F0F0Fu;
                so[T][1] = (k1[T] >> 4) & 0x0F0F0F0Fu;
            }
        } else {  // dword kk holds spread words 4kk..4kk+3; this lane's are 4kk + 2up (+1)
            const auto p0 = __builtin_amdgcn_permlane32_swap(c.c.x, c.c.x, false, false);
            const auto p1 = __builtin_amdgcn_permlane32_swap(c.c.y, c.c.y, false, false);
            const int sh = 4 * up;
#pragma unroll
            for (int T = 0; T < 2; ++T) {
                se[T][0] = (p0[T] >> sh) & 0x03030303u;
                so[T][0] = (p0[T] >> (sh + 2)) & 0x03030303u;
                se[T][1] = (p1[T] >> sh) & 0x03030303u;
                so[T][1] = (p1[T] >> (sh + 2)) & 0x03030303u;
            }
        }
        if constexpr (FB == 5 || FB == 3) {  // top bit of spread word s at bit s of each byte
            constexpr int top = FB == 5 ? 4 : 2;
            const auto hh = __builtin_amdgcn_permlane32_swap(c.h, c.h, false, false);
#pragma unroll
            for (int T = 0; T < 2; ++T)
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) {
                    const int sb = 4 * kk + 2 * up;
                    se[T][kk] |= ((hh[T] >> sb) & 0x01010101u) << top;
                    so[T][kk] |= ((hh[T] >> (sb + 1)) & 0x01010101u) << top;
                }
        }
    }
};

// The lane's NW metadata words of super-block slot si.
template <int NW>
__device__ __forceinline__ void load_words(const RplArgs& a, int64_t si, int lane, uint32_t* w) {
    if constexpr (NW == 2) {
        const uint2 v = reinterpret_cast<const uint2*>(a.meta)[si * 64 + lane];
        w[0] = v.x;
        w[1] = v.y;
    } else {
#pragma unroll
        for (int k = 0; k < NW / 4; ++k) {
            const uint4 v = ld_nt(reinterpret_cast<const uint4*>(a.meta) + (si * 64 + lane) * (NW / 4) + k);
            w[4 * k] = v.x;
            w[4 * k + 1] = v.y;
            w[4 * k + 2] = v.z;
            w[4 * k + 3] = v.w;
        }
    }
}

// Per-format B-operand builders of the GEMM kernels. Codes holds the code
// planes of one 32-column chunk of the lane's row and Meta the row's metadata
// of a whole super-block, loaded once for its 8 chunks (a word per chunk read
// with every chunk costs the L1 16 lines for 256 bytes, 8 times over); Ch is
// one chunk of both, j known at compile time, and load() a Ch read at once
// (k_gemm_q4k_pw, whose registers hold no super-block's metadata). k_gemm_rg
// takes Meta up to kMetaAhead 32-token tiles and a Ch per chunk beyond:
// records of 16 words cost it more registers than loads (TernaryPacked
// 4096->14336, 32 tokens, 21.1 us with Meta against 17.2, IQ3_S 64 tokens 27.0
// against 22.9, Q5_1 128 tokens 47.4 against 43.7), and of 8 words two or more
// tiles of the one-scale formats (BinaryPacked 14336->4096, 64 tokens, 27.9
// against 26.8) and four of Q5_K, Q3_K and IQ4_NL (4096->14336, 128 tokens, 43.8
// against 42.2 and 43.7 against 42.2), which load one word a chunk.
// bops() returns the fp16 B operands bf[T][kk] of 32-row tile T and k16 step
// kk, in X's k order [0,2,4,6,1,3,5,7], with the tile row's scales and mins
// multiplied by its power-of-two row factor wk[T] (RplArgs::wrow) before their
// fp16 cast.
// For the f32-precision batched forward (k_gemv_b), codes() gives the same
// operands as unscaled, exact fp16 code values (codes8) and scales() the f32
// scales of rows 32T + lane % 32: one per k16 step (kTwo) or one in kk = 0 per
// chunk, and with kMin the f32 offsets that meet the sums of x (or kMinBytes).
template <int FB>
struct GemmKQ {  // Q2_K, Q3_K, Q4_K, Q5_K: w = (d/255)*u*q + (dmin/127)*m
    static constexpr int kMetaAhead = FB == 2 || FB == 4 ? 4 : 2;
    struct Ch { typename GemmCodes<FB>::C c; uint32_t mw; float2 dd; };
    using Codes = typename GemmCodes<FB>::C;
    struct Meta { uint32_t w[8]; float2 dd; };
    static __device__ __forceinline__ Codes load_codes(const RplArgs& a, int64_t ci, int lane) {
        return GemmCodes<FB>::load(a, ci, lane);
    }
    static __device__ __forceinline__ Meta load_meta(const RplArgs& a, int64_t si, int lane) {
        Meta m;
        load_words<8>(a, si, lane, m.w);
        m.dd = reinterpret_cast<const float2*>(a.dd)[si * 64 + lane];
        return m;
    }
    static __device__ __forceinline__ Ch load(const RplArgs& a, int64_t ci, int64_t si, int j, int lane) {
        return {GemmCodes<FB>::load(a, ci, lane), reinterpret_cast<const uint32_t*>(a.meta)[(si * 64 + lane) * 8 + j],
                reinterpret_cast<const float2*>(a.dd)[si * 64 + lane]};
    }
    static __device__ __forceinline__ Ch chunk(const Codes& c, const Meta& m, int j) { return {c, m.w[j], m.dd}; }
    // The lane forms the fp16 scales and mins of its own row (row `lane` of
    // the group: tile lane / 32) and the lane swap hands each lane both tiles'
    // pairs, the same values the other lane computed.
    static __device__ __forceinline__ void bops(const Ch& c, int lane, const float (&wk)[2], half8 (&bf)[2][2]) {
        float w0 = wk[0], w1 = wk[1];
        asm("" : "+v"(w0), "+v"(w1));  // a select of values, not an indexed load of the array
        const float wo = (lane & 32) ? w1 : w0;  // the own row's factor
        const float d255 = c.dd.x * (wo * (1.0f / 255.0f)), dm127 = c.dd.y * (wo * (1.0f / 127.0f));
        const uint32_t gm = c.mw;
        const half2v scp = {_Float16(d255 * float(gm & 0xFFu)), _Float16(d255 * float((gm >> 8) & 0xFFu))};
        const half2v mnp = {_Float16(dm127 * float(int8_t(gm >> 16))), _Float16(dm127 * float(int32_t(gm) >> 24))};
        const auto sc2 = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, scp),
                                                          __builtin_bit_cast(uint32_t, scp), false, false);
        const auto mn2 = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, mnp),
                                                          __builtin_bit_cast(uint32_t, mnp), false, false);
        uint32_t se[2][2], so[2][2];
        GemmCodes<FB>::spread(c.c, lane, se, so);
#pragma unroll
        for (int T = 0; T < 2; ++T) {
            const half2v sp = __builtin_bit_cast(half2v, uint32_t(sc2[T])), np = __builtin_bit_cast(half2v, uint32_t(mn2[T]));
            const half2v s0 = {sp.x, sp.x}, s1 = {sp.y, sp.y}, n0 = {np.x, np.x}, n1 = {np.y, np.y};
            bf[T][0] = __builtin_bit_cast(half8, dequant8s<FB>(se[T][0], so[T][0], s0, n0));
            bf[T][1] = __builtin_bit_cast(half8, dequant8s<FB>(se[T][1], so[T][1], s1, n1));
        }
    }
    static constexpr bool kExact = true, kTwo = true, kMin = true;
    static __device__ __forceinline__ void codes(const Ch& c, int lane, half8 (&bf)[2][2]) {
        uint32_t se[2][2], so[2][2];
        GemmCodes<FB>::spread(c.c, lane, se, so);
        codes_all<FB, 0>(se, so, bf);
    }
    static __device__ __forceinline__ void scales(const Ch& c, float (&sc)[2][2], float (&mn)[2][2]) {
        const float d255 = c.dd.x * (1.0f / 255.0f);
        tile_rows(d255 * float(c.mw & 0xFFu), sc[0][0], sc[1][0]);
        tile_rows(d255 * float((c.mw >> 8) & 0xFFu), sc[0][1], sc[1][1]);
        (void)mn;
    }
    // The min bytes of the chunk's two groups as fp16 (own row), and per 32-row
    // tile the factor of their products with the group sums of x / 32.
    static constexpr bool kMinBytes = true;
    static __device__ __forceinline__ uint32_t min_codes(const Ch& c) {
        const half2v k1152 = {_Float16(1152.0f), _Float16(1152.0f)};
        const uint32_t u = __builtin_amdgcn_perm(0x64646464u, c.mw ^ 0x80800000u, 0x04030402u);  // 1024 + m + 128
        return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, u) - k1152);
    }
    static __device__ __forceinline__ void min_scale(const Meta& m, float (&dm)[2]) {
        tile_rows(m.dd.y * (32.0f / 127.0f), dm[0], dm[1]);
    }
};

struct GemmQ6 {  // Q6_K: q = lo4 | hi2 << 4, w = (d/255)*u*(q - 32)
    static constexpr int kMetaAhead = 4;
    struct Ch { uint4 c; uint2 h; uint32_t mw; float d; };
    struct Codes { uint4 c; uint2 h; };
    struct Meta { uint32_t w[4]; float d; };
    static __device__ __forceinline__ Codes load_codes(const RplArgs& a, int64_t ci, int lane) {
        return {ld_nt(reinterpret_cast<const uint4*>(a.codes) + ci * 64 + lane),
                reinterpret_cast<const uint2*>(a.hi)[ci * 64 + lane]};
    }
    static __device__ __forceinline__ Meta load_meta(const RplArgs& a, int64_t si, int lane) {
        Meta m;
        load_words<4>(a, si, lane, m.w);
        m.d = reinterpret_cast<const float*>(a.dd)[(si * 64 + lane) * 2];
        return m;
    }
    static __device__ __forceinline__ Ch load(const RplArgs& a, int64_t ci, int64_t si, int j, int lane) {
        const uint32_t m = reinterpret_cast<const uint32_t*>(a.meta)[(si * 64 + lane) * 4 + (j >> 1)];
        return {ld_nt(reinterpret_cast<const uint4*>(a.codes) + ci * 64 + lane),
                reinterpret_cast<const uint2*>(a.hi)[ci * 64 + lane], m >> (16 * (j & 1)),
                reinterpret_cast<const float*>(a.dd)[(si * 64 + lane) * 2]};
    }
    static __device__ __forceinline__ Ch chunk(const Codes& c, const Meta& m, int j) {
        return {c.c, c.h, m.w[j >> 1] >> (16 * (j & 1)), m.d};
    }
    // high-bit dword kk holds spread words 4kk..4kk+3 at bits 2f; this lane's are 4kk + 2up (+1)
    static __device__ __forceinline__ void spread6(const GemmCodes<4>::C& nib, uint2 h, int lane, uint32_t (&se)[2][2],
                                                   uint32_t (&so)[2][2]) {
        GemmCodes<4>::spread(nib, lane, se, so);
        const int sh = 4 * (lane >> 5);
        const auto h0 = __builtin_amdgcn_permlane32_swap(h.x, h.x, false, false);
        const auto h1 = __builtin_amdgcn_permlane32_swap(h.y, h.y, false, false);
#pragma unroll
        for (int T = 0; T < 2; ++T) {
            se[T][0] |= ((h0[T] >> sh) & 0x03030303u) << 4;
            so[T][0] |= ((h0[T] >> (sh + 2)) & 0x03030303u) << 4;
            se[T][1] |= ((h1[T] >> sh) & 0x03030303u) << 4;
            so[T][1] |= ((h1[T] >> (sh + 2)) & 0x03030303u) << 4;
        }
    }
    static __device__ __forceinline__ void bops(const Ch& c, int lane, const float (&wk)[2], half8 (&bf)[2][2]) {
        typename GemmCodes<4>::C nib{c.c, 0u};
        uint32_t se[2][2], so[2][2];
        spread6(nib, c.h, lane, se, so);
        // The own row's scales, handed to the tiles' lanes as one packed pair (as GemmKQ). Each is rounded once,
        // by the instruction that multiplies: as a conversion of two f32 products the pair is rounded twice, and a
        // block's outputs moved by 3.5e-6.
        float w0 = wk[0], w1 = wk[1];
        asm("" : "+v"(w0), "+v"(w1));
        const float d255 = c.d * (((lane & 32) ? w1 : w0) * (1.0f / 255.0f));
        uint32_t scp;
        asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(scp) : "v"(d255), "v"(float(c.mw & 0xFFu)));
        asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(scp) : "v"(d255), "v"(float((c.mw >> 8) & 0xFFu)));
        const auto sc2 = __builtin_amdgcn_permlane32_swap(scp, scp, false, false);
#pragma unroll
        for (int T = 0; T < 2; ++T) {
            const half2v k32 = {_Float16(-32.0f), _Float16(-32.0f)};
            const half2v sp = __builtin_bit_cast(half2v, uint32_t(sc2[T])), np = sp * k32;
            const half2v s0 = {sp.x, sp.x}, s1 = {sp.y, sp.y}, n0 = {np.x, np.x}, n1 = {np.y, np.y};
            bf[T][0] = __builtin_bit_cast(half8, dequant8s<6>(se[T][0], so[T][0], s0, n0));
            bf[T][1] = __builtin_bit_cast(half8, dequant8s<6>(se[T][1], so[T][1], s1, n1));
        }
    }
    static constexpr bool kExact = true, kTwo = true, kMin = false;
    static __device__ __forceinline__ void codes(const Ch& c, int lane, half8 (&bf)[2][2]) {
        typename GemmCodes<4>::C nib{c.c, 0u};
        uint32_t se[2][2], so[2][2];
        spread6(nib, c.h, lane, se, so);
        codes_all<6, 64>(se, so, bf);
    }
    static __device__ __forceinline__ void scales(const Ch& c, float (&sc)[2][2], float (&)[2][2]) {
        const float d255 = c.d * (1.0f / 255.0f);
        tile_rows(d255 * float(c.mw & 0xFFu), sc[0][0], sc[1][0]);
        tile_rows(d255 * float((c.mw >> 8) & 0xFFu), sc[0][1], sc[1][1]);
    }
};

struct GemmQ8 {  // Q8_0: w = scale*q, q int8, 32 bytes per chunk (consecutive columns)
    static constexpr int kMetaAhead = 4;
    struct Ch { uint4 c0, c1; uint32_t sc; };
    struct Codes { uint4 c0, c1; };
    struct Meta { uint32_t w[8]; };
    static __device__ __forceinline__ Codes load_codes(const RplArgs& a, int64_t ci, int lane) {
        const uint4* p = reinterpret_cast<const uint4*>(a.codes) + (ci * 64 + lane) * 2;
        return {ld_nt(p), ld_nt(p + 1)};
    }
    static __device__ __forceinline__ Meta load_meta(const RplArgs& a, int64_t si, int lane) {
        Meta m;
        load_words<8>(a, si, lane, m.w);
        return m;
    }
    static __device__ __forceinline__ Ch load(const RplArgs& a, int64_t ci, int64_t si, int j, int lane) {
        const uint4* p = reinterpret_cast<const uint4*>(a.codes) + (ci * 64 + lane) * 2;
        return {ld_nt(p), ld_nt(p + 1), reinterpret_cast<const uint32_t*>(a.meta)[(si * 64 + lane) * 8 + j]};
    }
    static __device__ __forceinline__ Ch chunk(const Codes& c, const Meta& m, int j) { return {c.c0, c.c1, m.w[j]}; }
    static __device__ __forceinline__ void bops(const Ch& c, int lane, const float (&wk)[2], half8 (&bf)[2][2]) {
        (void)lane;
        const uint32_t dw[8] = {c.c0.x, c.c0.y, c.c0.z, c.c0.w, c.c1.x, c.c1.y, c.c1.z, c.c1.w};
        const auto st = __builtin_amdgcn_permlane32_swap(c.sc, c.sc, false, false);
        const half2v k1152 = {_Float16(1152.0f), _Float16(1152.0f)};
        const uint32_t e = 0x64646464u;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            // lanes 0-31: columns 16kk + 0..7 (dwords 4kk, 4kk+1); lanes 32-63: + 8..15
            const auto A = __builtin_amdgcn_permlane32_swap(dw[4 * kk], dw[4 * kk + 2], false, false);
            const auto B = __builtin_amdgcn_permlane32_swap(dw[4 * kk + 1], dw[4 * kk + 3], false, false);
#pragma unroll
            for (int T = 0; T < 2; ++T) {
                const uint32_t lo = A[T] ^ 0x80808080u, hi = B[T] ^ 0x80808080u;  // q + 128 as unsigned bytes
                const uint32_t hb[4] = {__builtin_amdgcn_perm(e, lo, 0x04020400u), __builtin_amdgcn_perm(e, hi, 0x04020400u),
                                        __builtin_amdgcn_perm(e, lo, 0x04030401u), __builtin_amdgcn_perm(e, hi, 0x04030401u)};
                const _Float16 sh = _Float16(__uint_as_float(st[T]) * wk[T]);
                const half2v s2 = {sh, sh};
                uint32_t p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) p[i] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(half2v, hb[i]) - k1152) * s2);
                bf[T][kk] = __builtin_bit_cast(half8, make_uint4(p[0], p[1], p[2], p[3]));
            }
        }
    }
    static constexpr bool kExact = true, kTwo = false, kMin = false;
    static __device__ __forceinline__ void codes(const Ch& c, int lane, half8 (&bf)[2][2]) {
        (void)lane;
        const uint32_t dw[8] = {c.c0.x, c.c0.y, c.c0.z, c.c0.w, c.c1.x, c.c1.y, c.c1.z, c.c1.w};
        const half2v k1152 = {_Float16(1152.0f), _Float16(1152.0f)};
        const uint32_t e = 0x64646464u;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const auto A = __builtin_amdgcn_permlane32_swap(dw[4 * kk], dw[4 * kk + 2], false, false);
            const auto B = __builtin_amdgcn_permlane32_swap(dw[4 * kk + 1], dw[4 * kk + 3], false, false);
#pragma unroll
            for (int T = 0; T < 2; ++T) {
                const uint32_t lo = A[T] ^ 0x80808080u, hi = B[T] ^ 0x80808080u;
                const uint32_t hb[4] = {__builtin_amdgcn_perm(e, lo, 0x04020400u), __builtin_amdgcn_perm(e, lo, 0x04030401u),
                                        __builtin_amdgcn_perm(e, hi, 0x04020400u), __builtin_amdgcn_perm(e, hi, 0x04030401u)};
                uint32_t p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) p[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, hb[i]) - k1152);
                bf[T][kk] = __builtin_bit_cast(half8, make_uint4(p[0], p[1], p[2], p[3]));
            }
        }
    }
    static __device__ __forceinline__ void scales(const Ch& c, float (&sc)[2][2], float (&)[2][2]) {
        tile_rows(__uint_as_float(c.sc), sc[0][0], sc[1][0]);
    }
};

// The 32-weight block formats (Q4_0 with its nibble xor 8, Q4_1, Q5_0, Q5_1)
// and AffinePacked g64 (GSH = 1: chunks 2g, 2g+1 share group g): one scale
// (and min) per chunk from the lane's 8 (16) metadata words per super-block;
// w = scale*q + min, or scale*(q - OFF).
template <int FB, bool MIN, int OFF, uint32_t XR, int GSH = 0>
struct GemmB32 {
    static constexpr int NG = 8 >> GSH, NW = MIN ? 2 * NG : NG;
    static constexpr int kMetaAhead = NW <= 8 ? 4 : 0;
    struct Ch { typename GemmCodes<FB>::C c; uint32_t sc, mn; };
    using Codes = typename GemmCodes<FB>::C;
    struct Meta { uint32_t w[NW]; };
    static __device__ __forceinline__ Codes load_codes(const RplArgs& a, int64_t ci, int lane) {
        return GemmCodes<FB>::load(a, ci, lane);
    }
    static __device__ __forceinline__ Meta load_meta(const RplArgs& a, int64_t si, int lane) {
        Meta m;
        load_words<NW>(a, si, lane, m.w);
        return m;
    }
    static __device__ __forceinline__ Ch load(const RplArgs& a, int64_t ci, int64_t si, int j, int lane) {
        Ch r;
        r.c = GemmCodes<FB>::load(a, ci, lane);
        r.c.c.x ^= XR;
        r.c.c.y ^= XR;
        r.c.c.z ^= XR;
        r.c.c.w ^= XR;
        const uint32_t* m = reinterpret_cast<const uint32_t*>(a.meta) + (si * 64 + lane) * NW;
        r.sc = m[j >> GSH];
        r.mn = MIN ? m[NG + (j >> GSH)] : 0u;
        return r;
    }
    static __device__ __forceinline__ Ch chunk(const Codes& c, const Meta& m, int j) {
        Ch r{c, m.w[j >> GSH], MIN ? m.w[(NG + (j >> GSH)) % NW] : 0u};
        r.c.c.x ^= XR;
        r.c.c.y ^= XR;
        r.c.c.z ^= XR;
        r.c.c.w ^= XR;
        return r;
    }
    static __device__ __forceinline__ void bops(const Ch& c, int lane, const float (&wk)[2], half8 (&bf)[2][2]) {
        uint32_t se[2][2], so[2][2];
        GemmCodes<FB>::spread(c.c, lane, se, so);
        const auto st = __builtin_amdgcn_permlane32_swap(c.sc, c.sc, false, false);
        const auto mt = __builtin_amdgcn_permlane32_swap(c.mn, c.mn, false, false);
#pragma unroll
        for (int T = 0; T < 2; ++T) {
            const float scf = __uint_as_float(st[T]) * wk[T];
            const _Float16 sc = _Float16(scf), mn = _Float16(MIN ? __uint_as_float(mt[T]) * wk[T] : -float(OFF) * scf);
            const half2v s2 = {sc, sc}, n2 = {mn, mn};
            bf[T][0] = __builtin_bit_cast(half8, dequant8s<FB>(se[T][0], so[T][0], s2, n2));
            bf[T][1] = __builtin_bit_cast(half8, dequant8s<FB>(se[T][1], so[T][1], s2, n2));
        }
    }
    static constexpr bool kExact = true, kTwo = false, kMin = MIN;
    static __device__ __forceinline__ void codes(const Ch& c, int lane, half8 (&bf)[2][2]) {
        uint32_t se[2][2], so[2][2];
        GemmCodes<FB>::spread(c.c, lane, se, so);
        codes_all<FB, 2 * OFF>(se, so, bf);
    }
    static __device__ __forceinline__ void scales(const Ch& c, float (&sc)[2][2], float (&mn)[2][2]) {
        tile_rows(__uint_as_float(c.sc), sc[0][0], sc[1][0]);
        if constexpr (MIN) tile_rows(__uint_as_float(c.mn), mn[0][0], mn[1][0]);
    }
};

// Codes of one bit (BinaryPacked g32, IQ1_S): one word per chunk whose byte b
// holds at bit s the code of column 8(s/2) + 2b + s%2.
struct GemmCodes1 {
    struct C { uint32_t c; };
    static __device__ __forceinline__ C load(const RplArgs& a, int64_t ci, int lane) {
        return {reinterpret_cast<const uint32_t*>(a.codes)[ci * 64 + lane]};
    }
    static __device__ __forceinline__ void spread(const C& c, int lane, uint32_t (&se)[2][2], uint32_t (&so)[2][2]) {
        const auto hh = __builtin_amdgcn_permlane32_swap(c.c, c.c, false, false);
        const int up = lane >> 5;
#pragma unroll
        for (int T = 0; T < 2; ++T)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const int sb = 4 * kk + 2 * up;
                se[T][kk] = (hh[T] >> sb) & 0x01010101u;
                so[T][kk] = (hh[T] >> (sb + 1)) & 0x01010101u;
            }
    }
};

// The linear-code formats (the linear IQ formats, TernaryPacked, BinaryPacked
// g32 and g128): w = scale*(q - MID2/2), one scale per 32 columns, two (SG16,
// one per k16 step) or one per 2^GSH chunks; one-bit codes read +-scale =
// (2*scale)*(q - 1/2).
template <int FB, bool SG16, int MID2, int GSH = 0>
struct GemmLin {
    using Planes = std::conditional_t<FB == 1, GemmCodes1, GemmCodes<FB>>;
    static constexpr int NW = SG16 ? 16 : (8 >> GSH);  // metadata words per lane and super-block
    static constexpr int kMetaAhead = NW <= 8 ? 1 : 0;
    struct Ch { typename Planes::C c; uint32_t s0, s1; };
    using Codes = typename Planes::C;
    struct Meta { uint32_t w[NW]; };
    static __device__ __forceinline__ Codes load_codes(const RplArgs& a, int64_t ci, int lane) {
        return Planes::load(a, ci, lane);
    }
    static __device__ __forceinline__ Meta load_meta(const RplArgs& a, int64_t si, int lane) {
        Meta m;
        load_words<NW>(a, si, lane, m.w);
        return m;
    }
    static __device__ __forceinline__ Ch load(const RplArgs& a, int64_t ci, int64_t si, int j, int lane) {
        const uint32_t* m = reinterpret_cast<const uint32_t*>(a.meta) + (si * 64 + lane) * NW;
        const uint32_t s0 = m[SG16 ? 2 * j : (j >> GSH)];
        return {Planes::load(a, ci, lane), s0, SG16 ? m[2 * j + 1] : s0};
    }
    static __device__ __forceinline__ Ch chunk(const Codes& c, const Meta& m, int j) {
        const uint32_t s0 = m.w[SG16 ? 2 * j : (j >> GSH)];
        return {c, s0, SG16 ? m.w[(2 * j + 1) % NW] : s0};
    }
    static __device__ __forceinline__ void bops(const Ch& c, int lane, const float (&wk)[2], half8 (&bf)[2][2]) {
        uint32_t se[2][2], so[2][2];
        Planes::spread(c.c, lane, se, so);
        const auto t0 = __builtin_amdgcn_permlane32_swap(c.s0, c.s0, false, false);
        const auto t1 = __builtin_amdgcn_permlane32_swap(c.s1, c.s1, false, false);
        constexpr float mul = FB == 1 ? 2.0f : 1.0f, mid = 0.5f * MID2;
#pragma unroll
        for (int T = 0; T < 2; ++T)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const float scf = __uint_as_float(kk ? t1[T] : t0[T]) * (mul * wk[T]);
                const _Float16 sc = _Float16(scf), mn = _Float16(-mid * scf);
                const half2v s2 = {sc, sc}, n2 = {mn, mn};
                bf[T][kk] = __builtin_bit_cast(half8, dequant8s<FB>(se[T][kk], so[T][kk], s2, n2));
            }
    }
    static constexpr bool kExact = true, kTwo = SG16, kMin = false;
    static __device__ __forceinline__ void codes(const Ch& c, int lane, half8 (&bf)[2][2]) {
        uint32_t se[2][2], so[2][2];
        Planes::spread(c.c, lane, se, so);
        codes_all<FB, MID2>(se, so, bf);
    }
    static __device__ __forceinline__ void scales(const Ch& c, float (&sc)[2][2], float (&)[2][2]) {
        constexpr float mul = FB == 1 ? 2.0f : 1.0f;
        tile_rows(__uint_as_float(c.s0) * mul, sc[0][0], sc[1][0]);
        if constexpr (SG16) tile_rows(__uint_as_float(c.s1) * mul, sc[0][1], sc[1][1]);
    }
};

// IQ4_NL (quant/iq.go:169-180): w = scale * grid[q], the 16-value float grid
// (kIQ4NLGrid) as fp16, one scale per 32-column chunk. The codes are Q4_K's
// nibble planes; the grid is looked up four codes at a time with
// v_perm_b32 from byte tables of the fp16 values' low and high bytes (codes
// 0-7 from the first two dwords of a table, 8-15 from the last two, picked
// per byte by the code's bit 3), and the low and high bytes are interleaved
// into half2 pairs in k order [0,2,4,6,1,3,5,7].
struct GemmNL {
    static constexpr bool kExact = false;  // the float grid is not exact in fp16
    static constexpr uint16_t h16(int q) { return __builtin_bit_cast(uint16_t, _Float16(kIQ4NLGrid[q])); }
    static constexpr uint32_t tab(int n, int sh) {  // bytes 4n..4n+3 of the low (sh 0) or high (sh 8) table
        return uint32_t((h16(4 * n) >> sh) & 0xFF) | uint32_t((h16(4 * n + 1) >> sh) & 0xFF) << 8 |
               uint32_t((h16(4 * n + 2) >> sh) & 0xFF) << 16 | uint32_t((h16(4 * n + 3) >> sh) & 0xFF) << 24;
    }
    static constexpr int kMetaAhead = 2;
    struct Ch { GemmCodes<4>::C c; uint32_t s0; };
    using Codes = GemmCodes<4>::C;
    struct Meta { uint32_t w[8]; };
    static __device__ __forceinline__ Codes load_codes(const RplArgs& a, int64_t ci, int lane) {
        return GemmCodes<4>::load(a, ci, lane);
    }
    static __device__ __forceinline__ Meta load_meta(const RplArgs& a, int64_t si, int lane) {
        Meta m;
        load_words<8>(a, si, lane, m.w);
        return m;
    }
    static __device__ __forceinline__ Ch load(const RplArgs& a, int64_t ci, int64_t si, int j, int lane) {
        return {GemmCodes<4>::load(a, ci, lane), reinterpret_cast<const uint32_t*>(a.meta)[(si * 64 + lane) * 8 + j]};
    }
    static __device__ __forceinline__ Ch chunk(const Codes& c, const Meta& m, int j) { return {c, m.w[j]}; }
    // fp16 grid values of the 4 codes in the bytes of c: half2 of bytes 0, 1 and of bytes 2, 3
    static __device__ __forceinline__ void look4(uint32_t c, half2v& q01, half2v& q23) {
        constexpr uint32_t L0 = tab(0, 0), L1 = tab(1, 0), L2 = tab(2, 0), L3 = tab(3, 0);
        constexpr uint32_t H0 = tab(0, 8), H1 = tab(1, 8), H2 = tab(2, 8), H3 = tab(3, 8);
        const uint32_t sel = c & 0x07070707u;
        const uint32_t hi8 = ((c >> 3) & 0x01010101u) * 0xFFu;  // 0xFF in the bytes of codes 8-15
        const uint32_t lo = (__builtin_amdgcn_perm(L3, L2, sel) & hi8) | (__builtin_amdgcn_perm(L1, L0, sel) & ~hi8);
        const uint32_t hi = (__builtin_amdgcn_perm(H3, H2, sel) & hi8) | (__builtin_amdgcn_perm(H1, H0, sel) & ~hi8);
        q01 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(hi, lo, 0x05010400u));
        q23 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(hi, lo, 0x07030602u));
    }
    static __device__ __forceinline__ void bops(const Ch& c, int lane, const float (&wk)[2], half8 (&bf)[2][2]) {
        uint32_t se[2][2], so[2][2];
        GemmCodes<4>::spread(c.c, lane, se, so);
        const auto st = __builtin_amdgcn_permlane32_swap(c.s0, c.s0, false, false);
#pragma unroll
        for (int T = 0; T < 2; ++T) {
            const _Float16 sc = _Float16(__uint_as_float(st[T]) * wk[T]);
            const half2v s2 = {sc, sc};
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                half2v q[4];
                look4(se[T][kk], q[0], q[1]);
                look4(so[T][kk], q[2], q[3]);
                uint32_t p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) p[i] = __builtin_bit_cast(uint32_t, q[i] * s2);
                bf[T][kk] = __builtin_bit_cast(half8, make_uint4(p[0], p[1], p[2], p[3]));
            }
        }
    }
};

// The part of gemm_tiles.hip (gemm_tiles.h) that compiles a builder's kernels:
// two for each builder that takes longest (the second for its 256-token tiles),
// one for the linear codes and one for the rest.
template <class GP>
struct GemmPart : std::integral_constant<int, 7> {};
template <>
struct GemmPart<GemmKQ<3>> : std::integral_constant<int, 0> {};
template <>
struct GemmPart<GemmKQ<5>> : std::integral_constant<int, 2> {};
template <>
struct GemmPart<GemmQ6> : std::integral_constant<int, 4> {};
template <int FB, bool SG16, int MID2, int GSH>
struct GemmPart<GemmLin<FB, SG16, MID2, GSH>> : std::integral_constant<int, 6> {};
template <class GP>
constexpr int gemm_part(bool tall) {
    return GemmPart<GP>::value + (tall && GemmPart<GP>::value < 6 ? 1 : 0);
}

// Calls go.template run<GP>() with the B-operand builder of b's format.
template <class Go>
int with_builder(const DevBlob& b, const Go& go) {
    switch (b.fmt) {
    case FMT_Q2_K: go.template run<GemmKQ<2>>(); return 0;
    case FMT_Q3_K: go.template run<GemmKQ<3>>(); return 0;
    case FMT_Q4_K: go.template run<GemmKQ<4>>(); return 0;
    case FMT_Q5_K: go.template run<GemmKQ<5>>(); return 0;
    case FMT_Q6_K: go.template run<GemmQ6>(); return 0;
    case FMT_Q8_0: go.template run<GemmQ8>(); return 0;
    case FMT_Q4_0: go.template run<GemmB32<4, false, 8, 0x88888888u>>(); return 0;
    case FMT_Q4_1: go.template run<GemmB32<4, true, 0, 0u>>(); return 0;
    case FMT_Q5_0: go.template run<GemmB32<5, false, 16, 0u>>(); return 0;
    case FMT_Q5_1: go.template run<GemmB32<5, true, 0, 0u>>(); return 0;
    case FMT_AFFINE:
        switch (b.block_weights) {
        case 32: go.template run<GemmB32<4, true, 0, 0u, 0>>(); return 0;
        case 64: go.template run<GemmB32<4, true, 0, 0u, 1>>(); return 0;
        case 128: go.template run<GemmB32<4, true, 0, 0u, 2>>(); return 0;
        case 256: go.template run<GemmB32<4, true, 0, 0u, 3>>(); return 0;
        default: return int(hipErrorInvalidValue);
        }
    case FMT_BINARY:
        if (b.block_weights == 128) {
            go.template run<GemmLin<1, false, 1, 2>>();
            return 0;
        }
        [[fallthrough]];
    case FMT_IQ1_S: go.template run<GemmLin<1, false, 1>>(); return 0;
    case FMT_IQ2_XXS: go.template run<GemmLin<2, false, 3>>(); return 0;
    case FMT_IQ2_XS: go.template run<GemmLin<2, true, 3>>(); return 0;
    case FMT_IQ3_XXS: go.template run<GemmLin<3, false, 7>>(); return 0;
    case FMT_IQ3_S: go.template run<GemmLin<3, true, 7>>(); return 0;
    case FMT_IQ4_XS: go.template run<GemmLin<4, true, 15>>(); return 0;
    case FMT_TERNARY: go.template run<GemmLin<2, true, 2>>(); return 0;
    case FMT_IQ4_NL: go.template run<GemmNL>(); return 0;
    default: return int(hipErrorInvalidValue);
    }
}

}  // namespace
}  // namespace wv
