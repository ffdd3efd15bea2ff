// gemm_tiles.hip — the tile kernels of the prefill GEMM (gemm_rpl.hip has the
// operands, the conversions of X and the plans) and their launches. Compiled
// once per WV_GEMM_PART = 0 .. kGemmParts - 1.
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

constexpr int BK = 64;        // columns per K-step
constexpr int LDK = BK + 8;   // LDS row stride in halves (144 B: conflict-free 16 B row reads)

// Row factors (RplArgs::wrow) of row group g in the B-operand layout: wk[T]
// belongs to row 32T + lane % 32, the lane's row in 32-row tile T. Two plain
// loads rather than one and a lane swap: nothing waits for them before the
// first B operands (a swap right after the load would stall the wave for a
// memory round trip before its first code loads go out).
__device__ __forceinline__ void row_factors(const RplArgs& a, int g, int lane, float (&wk)[2]) {
    wk[0] = a.wrow[int64_t(g) * 64 + (lane & 31)];
    wk[1] = a.wrow[int64_t(g) * 64 + 32 + (lane & 31)];
}

// VALU instructions asked for after each MFMA of k_gemm_q4k_pw (0: the
// compiler's own order). The builders with two code planes make 6 to 7 per
// MFMA, which came out in runs of up to 100 between MFMAs. Measured, us, own
// order and as set: Q6_K 14336->4096 M = 509 91.6 / 89.5; Q5_K M = 512
// 4096->14336 96 / 84 (with 5: 91, with 9: 91), 14336->4096 100 / 96; Q3_K
// 4096->14336 85 / 81 (with 7: 85), 14336->4096 91 / 88. Q4_K and Q8_0, with
// fewer, ran slower with 4 (78.4 against 73.7 and 82.6 against 81.4 at M = 512).
template <class GP>
struct ValuPerMfma : std::integral_constant<int, 0> {};
template <>
struct ValuPerMfma<GemmQ6> : std::integral_constant<int, 4> {};
template <>
struct ValuPerMfma<GemmKQ<5>> : std::integral_constant<int, 7> {};
template <>
struct ValuPerMfma<GemmKQ<3>> : std::integral_constant<int, 9> {};

// Each of the 4 waves owns one 64-row group of the block's 256 rows and loads
// its row group's codes straight from the row-interleaved planes (lane l = row
// l, 16 bytes = 32 columns per chunk). One v_permlane32_swap per code-word
// pair turns that into MFMA B operands: after swapping words 0|1 (columns
// 0-7 | 8-15) between lanes l and l + 32, the first result holds rows 0-31
// with columns 0-7 in lanes 0-31 and 8-15 in lanes 32-63 (the 32x32x16 B
// layout of the first 32-row tile), the second the same for rows 32-63. Each
// wave dequantizes only its own rows (no copy shared through LDS), so the
// LDS carries X alone: per K-step a block writes 16 KB of fp16 X and each
// wave reads 16 KB back for 32 MFMAs (128 tokens x 64 rows x 64 columns),
// against 96 KB per 16 MFMAs per wave with fp16 W tiles.
// One wave per SIMD, so its LDS round trips are its own to hide: reading the A
// fragments a k16 step ahead (and X a step ahead of that, in three buffers)
// took Q4_K 4096->14336 from 81 to 75 us at M = 512, and 256-token tiles
// (TM = 8) from 302 to 268 at M = 2047; the register rings as named values or
// native vectors (the compiler kept a ring of structs in memory for Q8_0 and
// Q4_0) took Q8_0 M = 512 from 139 to 82, Q4_0 4096->4096 from 64 to 41. What
// bounds it now: 900 TFLOP/s at M = 2047, where the same loop without A reads
// and without dequantization runs 1060 and a register-only loop of these MFMAs
// on random data 1780 over 300 us (the clock gives way: 2150 over 2.5 ms);
// 448 tiles take two passes of 256 CUs.
template <class GP, int TM, int D, bool WF>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) k_gemm_q4k_pw(GemmArgs ga) {
    constexpr int BM = 32 * TM;
    constexpr int XB = BM * (BK / 8) / 256;  // 8-column X blocks per thread per K-step
    static_assert(XB >= 1 && 4 % D == 0, "shape");
    __shared__ __attribute__((aligned(16))) _Float16 xs[3][BM * LDK];
    __shared__ float xsc[BM];  // the tile's row factors, for the epilogue

    const RplArgs& a = ga.w;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // wave-uniform: chunk addresses stay scalar
    const int nblk = blockIdx.x, mblk = blockIdx.y, split = blockIdx.z;
    const int sb0 = split * ga.sb_per_split;
    const int sb1 = min(a.nsb, sb0 + ga.sb_per_split);
    const int steps = (sb1 - sb0) * 4;
    const int kb8 = ga.K / 8;
    // Row factors of the tile's tokens, staged once; the main loop's barriers
    // order these writes before the epilogue reads them.
    if (t < BM) xsc[t] = ga.xscale[min(mblk * BM + t, ga.M - 1)];
    const int g = min(nblk * 4 + wave, a.rg_count - 1);  // this wave's row group
    float wk[2] = {1.0f, 1.0f};  // row factors of the lane's rows in the two 32-row tiles
    if constexpr (WF) row_factors(a, g, lane, wk);

    struct Codes {
        typename GP::Ch c[2];  // the step's two chunks of this lane's row
    };
    struct Xv {
        u32x4 v[XB];  // fp16 X blocks of one K-step
    };
    auto load_c = [&](int s, Codes& r) {
        const int64_t si = int64_t(g) * a.nsb + sb0 + s / 4;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int j = 2 * (s & 3) + jj;
            r.c[jj] = GP::load(a, rpl_chunk(a, si, j), si, j, lane);
        }
    };
    // this thread's blocks: rows t / 8 + 32 i of the tile, block t % 8 of the step
    int xoff[XB];
#pragma unroll
    for (int i = 0; i < XB; ++i) xoff[i] = (min(mblk * BM + t / 8 + 32 * i, ga.M - 1) - mblk * BM) * kb8;
    const u32x4* xsrc = reinterpret_cast<const u32x4*>(ga.xh) + int64_t(mblk) * BM * kb8 + sb0 * 32 + t % 8;
    auto load_x = [&](int s) {
        Xv r;
#pragma unroll
        for (int i = 0; i < XB; ++i) r.v[i] = xsrc[xoff[i] + 8 * s];
        return r;
    };
    auto put_x = [&](int buf, const Xv& r) {
        _Float16* p = &xs[buf][(t / 8) * LDK + 8 * (t % 8)];
#pragma unroll
        for (int i = 0; i < XB; ++i) *reinterpret_cast<u32x4*>(p + 32 * i * LDK) = r.v[i];
    };
    auto read_a = [&](int buf, int ks, half8 (&af)[TM]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
            af[i] = *reinterpret_cast<const half8*>(&xs[buf][(i * 32 + (lane & 31)) * LDK + ks * 16 + 8 * (lane >> 5)]);
    };

    f32x16 acc[TM][2];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    Codes cr[D];
    // X of even and odd steps, in named registers: an indexed pair goes to memory
    Xv xa = load_x(0), xb = load_x(min(1, steps - 1));
#pragma unroll
    for (int d = 0; d < D; ++d) {
        load_c(min(d, steps - 1), cr[d]);
        __builtin_amdgcn_sched_barrier(0);
    }
    put_x(0, xa);
    put_x(1, xb);
    xa = load_x(min(2, steps - 1));
    if constexpr (TM < 8) xb = load_x(min(3, steps - 1));
    // B operands: [chunk][tile][k16 step] as fp16 in k order [0,2,4,6,1,3,5,7].
    // Step s + 1's are built (VALU) beside step s's MFMAs.
    half8 bf[2][2][2];
    GP::bops(cr[0].c[0], lane, wk, bf[0]);
    GP::bops(cr[0].c[1], lane, wk, bf[1]);
    load_c(min(D, steps - 1), cr[0]);
    __syncthreads();
    // One wave per SIMD: nothing else covers an LDS round trip, so the A
    // fragments of each k16 step are read one k16 step ahead, across the step
    // boundary too: X sits in three buffers (step s reads s and s + 1 and
    // writes s + 2, whose readers of step s - 1 the last barrier has passed).
    half8 a0[TM], a1[TM];
    read_a(0, 0, a0);
    int b0 = 0, b1 = 1, b2 = 2;  // buffers of steps s, s + 1, s + 2
    auto mfmas = [&](const half8 (&af)[TM], const half8 (&b)[2][2], int kk) {
        __builtin_amdgcn_sched_barrier(0x6);  // VALU and SALU may cross
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int T = 0; T < 2; ++T)
                acc[i][T] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], b[T][kk], acc[i][T], 0, 0, 0);
        if constexpr (ValuPerMfma<GP>::value > 0) {
#pragma unroll
            for (int i = 0; i < 2 * TM; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, ValuPerMfma<GP>::value, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0x6);
    };
    auto step = [&](auto E, int s) {
        constexpr int e = decltype(E)::value;
        Codes& c = cr[(e + 1) % D];
        half8 bn[2][2][2];  // step s + 1
        read_a(b0, 1, a1);
        if constexpr (TM == 8) {
            put_x(b2, xa);
            xa = load_x(min(s + 3, steps - 1));
        } else if constexpr (e & 1) {
            put_x(b2, xb);
            xb = load_x(min(s + 4, steps - 1));
        } else {
            put_x(b2, xa);
            xa = load_x(min(s + 4, steps - 1));
        }
        mfmas(a0, bf[0], 0);
        read_a(b0, 2, a0);
        GP::bops(c.c[0], lane, wk, bn[0]);
        mfmas(a1, bf[0], 1);
        read_a(b0, 3, a1);
        GP::bops(c.c[1], lane, wk, bn[1]);
        load_c(min(s + 1 + D, steps - 1), c);
        mfmas(a0, bf[1], 0);
        read_a(b1, 0, a0);
        mfmas(a1, bf[1], 1);
        __syncthreads();
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int T = 0; T < 2; ++T)
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) bf[jj][T][kk] = bn[jj][T][kk];
        const int bt = b0;
        b0 = b1;
        b1 = b2;
        b2 = bt;
    };
    for (int s0 = 0; s0 < steps; s0 += 4) {
        step(std::integral_constant<int, 0>{}, s0);
        step(std::integral_constant<int, 1>{}, s0 + 1);
        step(std::integral_constant<int, 2>{}, s0 + 2);
        step(std::integral_constant<int, 3>{}, s0 + 3);
    }

    // C[i][j] of a 32x32 tile: lane holds j = lane % 32, i = 8*(r/4) + 4*(lane/32) + r%4.
    float* out = ga.y + int64_t(split) * ga.M * a.rows;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int T = 0; T < 2; ++T) {
            const int n = (nblk * 4 + wave) * 64 + T * 32 + (lane & 31);
            if (n >= a.rows) continue;
            const float wi = WF ? 1.0f / wk[T] : 1.0f;  // the row factor back out (exact: a power of two)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = mblk * BM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m < ga.M) out[int64_t(m) * a.rows + n] = acc[i][T][r] * wi * xsc[m - mblk * BM];
            }
        }
}

// The token-block GEMM for few tokens (TM 32-token tiles, TM = 1 or 2): one
// block per (64-row group, token block, K split), its W waves splitting the
// split's super-blocks (`per` consecutive ones each). A wave loads its row
// group's codes from the planes as k_gemm_q4k_pw does (B operands through
// lane swaps) and its fp16 X fragments straight from global memory (one
// contiguous 1 KB per wave and load: the A-fragment order of GemmArgs::xh),
// so the main loop has no barrier and no LDS traffic. A step is 64 columns
// (two chunks, four k16 MFMA steps); codes run DC steps ahead of use and X
// fragments (L2 hits: every row group's blocks read the same X) DX steps
// ahead, in register rings. A super-block's metadata comes in whole one
// super-block ahead where GP::kMetaAhead says so (word by word with each chunk,
// its 4-byte loads at a 32-byte stride filled the L1: Q4_K 4096->14336 M = 32
// 19.5 against 21.2 us, 4096->4096 17.1 against 18.2), else with each chunk.
// Every weight is dequantized once per token block.
// The W waves' partial tiles meet in LDS after the loop and are added in wave
// order (deterministic), one 32-token tile at a time.
template <class GP, int TM, int DC, int DX, int NT, bool WF>
__global__ void __launch_bounds__(NT) k_gemm_rg(GemmArgs ga, int per) {
    constexpr int BM = 32 * TM;
    static_assert(4 % DC == 0 && 4 % DX == 0, "the rings must divide the 4 steps of a super-block");
    constexpr bool kAhead = TM <= GP::kMetaAhead;  // metadata a super-block ahead, else with each chunk
    constexpr int DU = kAhead ? 4 : DC > DX ? DC : DX;  // loop unroll: ring positions (and metadata words) are compile-time
    extern __shared__ float red[];  // [W][2][16][64] partial tiles of one 32-token tile
    const RplArgs& a = ga.w;
    const int t = threadIdx.x, lane = t & 63, W = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // wave-uniform: chunk addresses stay scalar
    const int g = blockIdx.x, mblk = blockIdx.y, split = blockIdx.z;
    const int sb0 = split * ga.sb_per_split;
    const int sb1 = min(a.nsb, sb0 + ga.sb_per_split);
    const int wsb0 = sb0 + wave * per;
    const int steps = max(0, min(sb1, wsb0 + per) - wsb0) * 4;
    const int mt = (ga.M + 31) / 32;  // 32-token tiles of the fragment-ordered X
    float wk[2] = {1.0f, 1.0f};  // row factors of the lane's rows in the two 32-row tiles
    if constexpr (WF) row_factors(a, g, lane, wk);

    struct Codes {
        std::conditional_t<kAhead, typename GP::Codes, typename GP::Ch> c[2];  // the step's two chunks of this lane's row
    };
    struct Xf {
        uint4 v[TM][4];  // A fragments of the step's 4 k16 steps
    };
    auto load_c = [&](int s, Codes& r) {
        const int64_t si = int64_t(g) * a.nsb + wsb0 + s / 4;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int j = 2 * (s & 3) + jj;
            if constexpr (kAhead) r.c[jj] = GP::load_codes(a, rpl_chunk(a, si, j), lane);
            else r.c[jj] = GP::load(a, rpl_chunk(a, si, j), si, j, lane);
        }
    };
    auto load_m = [&](int sb) { return GP::load_meta(a, int64_t(g) * a.nsb + wsb0 + sb, lane); };
    auto load_x = [&](int s, Xf& r) {
        const int64_t q0 = int64_t(wsb0) * 16 + 4 * s;  // first k16 step of the step
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) r.v[i][ks] = ga.xh[((q0 + ks) * mt + mblk * TM + i) * 64 + lane];
    };

    f32x16 acc[TM][2];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    if (steps > 0) {
        Codes cr[DC];
        Xf xr[DX];
        [[maybe_unused]] typename GP::Meta mt, mnext;
        if constexpr (kAhead) mnext = load_m(0);
#pragma unroll
        for (int d = 0; d < (DC > DX ? DC : DX); ++d) {
            if (d < DC) load_c(min(d, steps - 1), cr[d % DC]);
            if (d < DX) load_x(min(d, steps - 1), xr[d % DX]);
            __builtin_amdgcn_sched_barrier(0);
        }
        for (int s0 = 0; s0 < steps; s0 += DU) {
            if constexpr (kAhead) {
                mt = mnext;
                mnext = load_m(min(s0 + 4, steps - 4) / 4);
            }
#pragma unroll
            for (int d = 0; d < DU; ++d) {
                const int s = s0 + d;
                const Codes cc = cr[d % DC];
                const Xf xc = xr[d % DX];
                __builtin_amdgcn_sched_barrier(0);
                load_c(min(s + DC, steps - 1), cr[d % DC]);
                load_x(min(s + DX, steps - 1), xr[d % DX]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    half8 bf[2][2];  // [tile][k16 step]
                    if constexpr (kAhead) GP::bops(GP::chunk(cc.c[jj], mt, 2 * d + jj), lane, wk, bf);
                    else GP::bops(cc.c[jj], lane, wk, bf);
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                        for (int i = 0; i < TM; ++i) {
                            const half8 af = __builtin_bit_cast(half8, xc.v[i][2 * jj + kk]);
#pragma unroll
                            for (int T = 0; T < 2; ++T)
                                acc[i][T] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf[T][kk], acc[i][T], 0, 0, 0);
                        }
                }
            }
        }
    }

    // C[i][j] of a 32x32 tile: lane holds j = lane % 32, i = 8*(r/4) + 4*(lane/32) + r%4.
    float* out = ga.y + int64_t(split) * ga.M * a.rows;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        if (i > 0) __syncthreads();  // the previous tile's sums have been read
#pragma unroll
        for (int T = 0; T < 2; ++T) {
            const float wi = WF ? 1.0f / wk[T] : 1.0f;  // the row factor back out (exact: a power of two)
#pragma unroll
            for (int r = 0; r < 16; ++r) red[((wave * 2 + T) * 16 + r) * 64 + lane] = acc[i][T][r] * wi;
        }
        __syncthreads();
        for (int v = t; v < 2048; v += 64 * W) {
            const int T = v >> 10, r = (v >> 6) & 15, l = v & 63;
            float sum = 0.f;
            for (int w = 0; w < W; ++w) sum += red[((w * 2 + T) * 16 + r) * 64 + l];
            const int n = g * 64 + T * 32 + (l & 31);
            const int m = mblk * BM + i * 32 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3);
            if (n < a.rows && m < ga.M) out[int64_t(m) * a.rows + n] = sum * ga.xscale[m];
        }
    }
}

// k_gemm_q4k_pw with TM 32-token tiles per wave; WF: apply the row factors.
template <int TM, bool WF>
struct PwGo {
    dim3 grid;
    hipStream_t s;
    const GemmArgs& ga;
    template <class GP>
    void run() const {
        if constexpr (gemm_part<GP>(TM == 8) == WV_GEMM_PART)
            hipLaunchKernelGGL((k_gemm_q4k_pw<GP, TM, TM == 8 ? 2 : 4, WF>), grid, dim3(256), 0, s, ga);
    }
};

// k_gemm_rg with TM token tiles per block, `per` super-blocks per wave, W
// waves (at most rg_waves(TM)). Ring depths and block size per token tiles:
// one or two tiles run 8 waves (2 per SIMD, 256 registers each), four tiles 4
// waves (1 per SIMD, whose 512 registers hold the 128 accumulators and deeper
// rings).
template <int TM, bool WF>
struct RgGo {
    dim3 grid;
    int W, per;
    hipStream_t s;
    const GemmArgs& ga;
    template <class GP>
    void run() const {
        if constexpr (gemm_part<GP>(false) == WV_GEMM_PART) {
            constexpr int DC = TM == 2 ? 2 : 4, DX = TM == 1 ? 2 : TM == 2 ? 1 : 2, NT = TM == 4 ? 256 : 512;
            const size_t lds = size_t(W) * 2 * 16 * 64 * sizeof(float);
            hipLaunchKernelGGL((k_gemm_rg<GP, TM, DC, DX, NT, WF>), grid, dim3(unsigned(64 * W)), lds, s, ga, per);
        }
    }
};

template <bool WF>
int launch_tiles(const DevBlob& b, const GemmPlan& p, dim3 grid, hipStream_t s, const GemmArgs& ga) {
    if (p.kind == GEMM_RG)
        return p.bm == 32   ? with_builder(b, RgGo<1, WF>{grid, p.W, p.per, s, ga})
               : p.bm == 64 ? with_builder(b, RgGo<2, WF>{grid, p.W, p.per, s, ga})
                            : with_builder(b, RgGo<4, WF>{grid, p.W, p.per, s, ga});
    return p.bm == 256 ? with_builder(b, PwGo<8, WF>{grid, s, ga}) : with_builder(b, PwGo<4, WF>{grid, s, ga});
}
}  // namespace

template <int PART>
int launch_gemm_tiles(const DevBlob& b, const GemmPlan& p, dim3 grid, hipStream_t s, const GemmArgs& ga) {
    return b.gemm_row_factors ? launch_tiles<true>(b, p, grid, s, ga) : launch_tiles<false>(b, p, grid, s, ga);
}
template int launch_gemm_tiles<WV_GEMM_PART>(const DevBlob&, const GemmPlan&, dim3, hipStream_t, const GemmArgs&);

}  // namespace wv
