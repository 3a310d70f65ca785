// Prefill dequant-GEMM for few rows: Y[M tokens, N rows] (+)= X[M,K] * W[N,K]^T
// over the messages, chat turns and default-sized chunks (up to a few hundred
// tokens) whose grids of 64x64 tiles leave most of the chip idle.
//
// What bounds these products is latency: a layer's projection is 0.3-3 MB of
// weights and well under a microsecond of the chip's matrix cores, but a
// pipelined tile (dgemm_kernel) walks K at a memory round trip per 64-wide
// stage, 9 to 24 of them for K = 576 to 1,536, on 15 to 120 workgroups.  Here
// a workgroup of NW waves owns a small output tile (16 TM x 16 TN per matrix)
// and its waves split K: each takes a contiguous share of the 64-wide stages
// and moves them by DMA into LDS stage buffers of its own, D stages in flight,
// so that no wave waits for another until the accumulators meet in LDS at the
// end.  (Loading the MFMA fragments straight into registers instead puts every
// lane on a row of its own, and the address unit then serves one lane per
// clock: 4x slower per byte than the DMA's 64-byte runs.)
//
// The RMSNorm in front of QKV and gate/up is part of the kernel (NV > 0): a
// workgroup reads whole rows of its activations anyway, as float32 (the bytes
// of two f16 terms), so while the weights are on their way each wave
// normalises some of the tile's rows, as rmsnorm_rows_kernel does, and leaves
// their f16 terms in LDS for all waves.
//
// Arithmetic as in dgemm_kernel: weights enter as their exact integer quants,
// activations as one f16 term or two (hi + lo) in the tiles from lo_row0 on,
// and each block's float32 MFMA result is scaled by d before it is added.
// Each wave adds its blocks in K order and the waves' sums are added in wave
// order, so an output depends on K and NW only, not on the tile or the grid.
//
// F32 (calls of 2 to 15 tokens): float32 activations without loss.  A float32 is
// the exact sum of three bf16 terms (24 significant bits in three times 8, the
// exponent range the same; below 2^-102 the last ones are subnormal and may be
// lost, 2^-126 at most), a quant or nibble is one and an f16 weight two, so
// bf16 MFMA products of the terms are the float32 products themselves, summed in
// float32, smallest terms first.  The rows stay float32 in HBM and LDS (the bytes
// of two f16 terms) and a lane takes a fragment apart as it reads it: with K split
// over the waves each element is taken apart once a workgroup.  (An infinity gives
// NaN one product earlier than the next RMSNorm would.)  Of a layer whose logits
// pass gate+up, down and the head, relative to 64 bits: 1.8e-7 to 2.5e-7 at every
// shape and format below, for rows from 1e-3 and products from 1e-6 to past 65,504;
// the float32 GEMM on the VALU 2.7e-7 to 4.3e-7 (Q8_0, Q4_0) and 0.9e-6 to 2.0e-6
// (F16).  11 rows, us a launch, VALU / this (QKV and gate+up of the first two with
// their RMSNorm, another 2.7 before the VALU's):
//   135M shape, Q8_0   QKV  5.3 / 5.8   Wo  5.2 / 4.1   gate+up 11.7 /  6.2   down  8.4 /  5.2
//   360M shape, Q4_0   QKV  6.7 / 6.6   Wo  5.2 / 4.7   gate+up 14.1 /  7.5   down 10.2 /  7.0
//   1.7B shape, Q8_0   QKV 28.0 / 8.9   Wo 18.3 / 6.3   gate+up 57.0 / 13.6   down 59.2 / 14.0
#include "common.h"
#include "gemm_frag.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

namespace {

struct SmallArgs {
    SmallGemmInput in;
    int M;
    DevMatrix w, u;
    float* y;
    f16* yh;
    f16* yhlo;
    int ldy;
    int lo_row0, lo_out_row0, lo_col0;
    int by_cols;  // tiles column by column (else row by row), XCD-major
    QkvRope qkv;
};

constexpr int SK = 64;  // K per stage (two quant blocks)
constexpr int kNormV = 4;  // float4 per lane of a normalised row (K <= 1,024)

// One wave's stage buffer: the activations' rows (128 B, the second term's
// after the first's, or 256 B of float32; absent with NORM, whose rows are
// shared), each matrix's weight rows, each matrix's scale pairs.
template <int FMT, int TM, int TN, int NB, bool NORM, bool F32>
struct SmallStage {
    static constexpr int BROW = FMT == DT_Q8_0 ? 64 : FMT == DT_Q4_0 ? 32 : 128;
    static constexpr int A_LO = 16 * TM * 128;
    static constexpr int B_OFF = NORM ? 0 : 2 * A_LO;
    static constexpr int S_OFF = B_OFF + NB * 16 * TN * BROW;
    static constexpr int BYTES = S_OFF + (FMT == DT_F16 ? 0 : NB * 16 * TN * 4);
    // DMA instructions of a stage, without the activations' second term
    static constexpr int B_I = FMT == DT_Q8_0 ? TN : FMT == DT_Q4_0 ? (TN + 1) / 2 : 2 * TN;
    static constexpr int A_I = NORM ? 0 : F32 ? 4 * TM : 2 * TM;
    static constexpr int PER = A_I + NB * (B_I + (FMT == DT_F16 ? 0 : 1));
};

// LDS row pitch of the normalised activations: 16 bytes past a multiple of 256,
// so the 16 rows of a fragment read fall in 16 distinct 16-byte bank groups.
__host__ __device__ constexpr int norm_pitch(int row_bytes) { return (row_bytes + 255) / 256 * 256 + 16; }

// Bytes of the tile's normalised rows: two f16 planes or one of float32.
template <int TM, bool F32>
__host__ __device__ constexpr int norm_bytes(int K) {
    return 16 * TM * (F32 ? norm_pitch(4 * K) : 2 * norm_pitch(2 * K));
}

template <int FMT, int MODE, int TM, int TN, int NW, int D, int NV, bool F32>
constexpr size_t small_lds(int K) {
    constexpr int NB = MODE == GEMM_SWIGLU ? 2 : 1;
    const size_t ring = (size_t)NW * D * SmallStage<FMT, TM, TN, NB, (NV > 0), F32>::BYTES;
    const size_t rows = NV > 0 ? (size_t)norm_bytes<TM, F32>(K) : 0;
    return std::max(ring + rows, (size_t)NW * NB * TM * TN * 1024);  // the waves' accumulators reuse it
}

// The top halves of two floats as a bf16 pair.
__device__ __forceinline__ uint32_t bf16_tops(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float bf16_top(float a) { return __uint_as_float(__float_as_uint(a) & 0xFFFF0000u); }
__device__ __forceinline__ bf16x8 as_bf16x8(const uint32_t (&o)[4]) {
    return __builtin_bit_cast(bf16x8, make_uint4(o[0], o[1], o[2], o[3]));
}
// Eight floats as N bf16 terms, largest first: each the top half of what the ones
// before it leave (exact differences; three hold a float32 from 2^-102 on, two
// every f16).
template <int N>
__device__ __forceinline__ void bf16_split(float (&x)[8], bf16x8 (&t)[N]) {
#pragma unroll
    for (int n = 0; n < N; n++) {
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = bf16_tops(x[2 * e], x[2 * e + 1]);
        t[n] = as_bf16x8(o);
        if (n + 1 < N)
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] -= bf16_top(x[e]);
    }
}

template <int FMT, int MODE, int TM, int TN, int NW, int D, int NV, bool F32>
__global__ __launch_bounds__(64 * NW) void small_gemm_kernel(SmallArgs p) {
    constexpr int NB = MODE == GEMM_SWIGLU ? 2 : 1;
    constexpr int F = TM * TN;  // 16x16 fragments per matrix
    constexpr bool QUANT = FMT != DT_F16, NORM = NV > 0;
    using L = SmallStage<FMT, TM, TN, NB, NORM, F32>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const int K = p.w.cols, N = p.w.rows, M = p.M, nb = K >> 5, nk = K / SK, spitch = stage_scale_pitch(N);
    const int tiles_m = (M + 16 * TM - 1) / (16 * TM), tiles_n = (N + 16 * TN - 1) / (16 * TN);
    const int tiles = tiles_m * tiles_n, xcd = blockIdx.x % 8, tq = tiles / 8, rem = tiles % 8;
    const int t = xcd * tq + min(xcd, rem) + blockIdx.x / 8;  // XCD-major (bijective)
    const int tm_i = p.by_cols ? t % tiles_m : t / tiles_n, tn_i = p.by_cols ? t / tiles_m : t % tiles_n;
    const int m0 = tm_i * 16 * TM, n0 = tn_i * 16 * TN;
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int per = (nk + NW - 1) / NW, k0 = wave * per, cnt = max(0, min(nk - k0, per));  // this wave's stages
    const bool use_lo = (NORM || p.in.xlo) && (m0 + 16 * TM > p.lo_row0 || n0 + 16 * TN > p.lo_col0);
    const int pitch = norm_pitch(F32 ? 4 * K : 2 * K);
    uint8_t* const rows = smem;  // NORM: the tile's normalised rows, first terms then second, or float32
    uint8_t* const ring = smem + (NORM ? norm_bytes<TM, F32>(K) : 0) + wave * D * L::BYTES;

    // Per-lane DMA source offsets (rows past the edges clamped to the last).
    uint32_t aoff[NORM ? 1 : L::A_I], boff[L::B_I], soff = 0;
    if constexpr (!NORM) {
#pragma unroll
        for (int i = 0; i < L::A_I; i++) {
            if constexpr (F32) {
                const int r = 4 * i + (lane >> 4), c = (lane & 15) ^ (r & 15);
                aoff[i] = (uint32_t)((min(m0 + r, M - 1) * p.in.ldx + c * 4) * 4);
            } else {
                const int r = 8 * i + (lane >> 3), c = (lane & 7) ^ swz_a(r);
                aoff[i] = (uint32_t)((min(m0 + r, M - 1) * p.in.ldx + c * 8) * 2);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < L::B_I; i++) {
        if constexpr (FMT == DT_Q8_0) {
            const int r = 16 * i + (lane >> 2), c = (lane & 3) ^ swz_q8(r);
            boff[i] = (uint32_t)(min(n0 + r, N - 1) * K + c * 16);
        } else if constexpr (FMT == DT_Q4_0) {
            const int r = 32 * i + (lane >> 1), c = (lane & 1) ^ swz_q4(r);
            boff[i] = (uint32_t)((min(n0 + r, N - 1) * nb + c) * 16);
        } else {
            const int r = 8 * i + (lane >> 3), c = (lane & 7) ^ swz_a(r);
            boff[i] = (uint32_t)((min(n0 + r, N - 1) * K + c * 8) * 2);
        }
    }
    if constexpr (QUANT) soff = (uint32_t)(min(n0 + lane, N - 1) * 4);

    // Stage kt into the stage buffer at LDS address sg.
    auto issue = [&](uint32_t sg_, int kt_, auto tt_c) {
        constexpr bool TT = decltype(tt_c)::value;
        // (wave-uniform: the DMA takes its base and its LDS address in SGPRs)
        const uint32_t sg = __builtin_amdgcn_readfirstlane(sg_);
        const int kt = __builtin_amdgcn_readfirstlane(kt_);
        if constexpr (!NORM) {
#pragma unroll
            for (int i = 0; i < L::A_I; i++) {
                if constexpr (F32) dma16s(p.in.xf + kt * SK, aoff[i], sg + i * 1024);
                else dma16s(p.in.x + kt * SK, aoff[i], sg + i * 1024);
                if constexpr (TT) dma16s(p.in.xlo + kt * SK, aoff[i], sg + L::A_LO + i * 1024);
            }
        }
#pragma unroll
        for (int mat = 0; mat < NB; mat++) {
            const DevMatrix& w = mat ? p.u : p.w;
            const uint32_t bq = sg + L::B_OFF + mat * 16 * TN * L::BROW;
#pragma unroll
            for (int i = 0; i < L::B_I; i++) {
                if constexpr (FMT == DT_Q8_0) {
                    dma16s(w.q + kt * SK, boff[i], bq + i * 1024);
                } else if constexpr (FMT == DT_Q4_0) {
                    if (32 * i + (lane >> 1) < 16 * TN) dma16s(w.q + kt * 32, boff[i], bq + i * 1024);
                } else {
                    dma16s(w.q + kt * SK * 2, boff[i], bq + i * 1024);
                }
            }
            if constexpr (QUANT) {
                const uint32_t* sc = w.s2 + (uint32_t)(kt * spitch);
                if (lane < 16 * TN) dma4s(sc, soff, sg + L::S_OFF + mat * 16 * TN * 4);
            }
        }
    };

    f32x4 acc[NB][TM][TN];
#pragma unroll
    for (int mat = 0; mat < NB; mat++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[mat][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // The fragments this wave finishes (f = wave, wave + NW, ...).  What their
    // epilogue reads (the residual, the RoPE pairs) is loaded with the operands.
    constexpr int FW = (F + NW - 1) / NW;
    float pre[FW][4][2];
#pragma unroll
    for (int k = 0; k < FW; k++) {
        const int f = wave + k * NW;
        if (f >= F) break;
        const int mb = m0 + 16 * (f / TN) + 4 * g, n = min(n0 + 16 * (f % TN) + l16, N - 1);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = min(mb + r, M - 1);
            if constexpr (MODE == GEMM_ACC) pre[k][r][0] = p.y[(int64_t)m * p.ldy + n];
            if constexpr (MODE == GEMM_QKV_ROPE) {
                const float2 cs = p.qkv.rope[(int64_t)(p.qkv.pos + m) * (p.qkv.hd / 2) + (n % p.qkv.hd) / 2];
                pre[k][r][0] = cs.x;
                pre[k][r][1] = cs.y;
            }
        }
    }

    auto run = [&](auto tt_c) {
        constexpr bool TT = decltype(tt_c)::value;
        constexpr int PER = L::PER + (TT ? L::A_I : 0);
        static_assert((D - 1) * PER < 64, "vmcnt range");
        auto compute = [&](const uint8_t* sg, int kt) {
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                f16x8 ah[TM], al[TT ? TM : 1];
                bf16x8 ax[F32 ? TM : 1][3];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const int r = 16 * i + l16;
                    if constexpr (F32) {
                        float xv[8];
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const uint8_t* a =
                                NORM ? rows + r * pitch + (kt * SK + 32 * kk + 8 * g + 4 * h) * 4
                                     : sg + r * 256 + ((8 * kk + 2 * g + h) ^ (r & 15)) * 16;
                            const f32x4 v = *(const f32x4*)a;
#pragma unroll
                            for (int e = 0; e < 4; e++) xv[4 * h + e] = v[e];
                        }
                        bf16_split(xv, ax[i]);
                    } else if constexpr (NORM) {
                        const uint8_t* a = rows + r * pitch + (kt * SK + 32 * kk + 8 * g) * 2;
                        ah[i] = *(const f16x8*)a;
                        if constexpr (TT) al[i] = *(const f16x8*)(a + 16 * TM * pitch);
                    } else {
                        const int o = r * 128 + ((4 * kk + g) ^ swz_a(r)) * 16;
                        ah[i] = *(const f16x8*)(sg + o);
                        if constexpr (TT) al[i] = *(const f16x8*)(sg + L::A_LO + o);
                    }
                }
#pragma unroll
                for (int mat = 0; mat < NB; mat++)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        const int r = 16 * j + l16;
                        const uint8_t* bq = sg + L::B_OFF + mat * 16 * TN * L::BROW;
                        f16x8 bf;
                        bf16x8 bx[FMT == DT_F16 ? 2 : 1];
                        float d = 1.f;
                        if constexpr (QUANT) {
                            uint32_t o[4];
                            if constexpr (FMT == DT_Q8_0) {
                                const int u = 4 * kk + g;
                                const uint2 raw = *(const uint2*)(bq + r * 64 + ((u >> 1) ^ swz_q8(r)) * 16 + (u & 1) * 8);
                                if constexpr (F32) {
                                    int8x4_to_bf16(raw.x, o[0], o[1]);
                                    int8x4_to_bf16(raw.y, o[2], o[3]);
                                } else {
                                    int8x4_to_f16(raw.x, o[0], o[1]);
                                    int8x4_to_f16(raw.y, o[2], o[3]);
                                }
                            } else {
                                const uint2 raw = *(const uint2*)(bq + r * 32 + (kk ^ swz_q4(r)) * 16 + (g & 1) * 8);
                                const int sh = (g >> 1) * 4;  // low nibbles: elements 0..15, high: 16..31
                                const uint32_t n0_ = (raw.x >> sh) & 0x0F0F0F0Fu, n1_ = (raw.y >> sh) & 0x0F0F0F0Fu;
                                if constexpr (F32) {
                                    nib4_to_bf16(n0_, o[0], o[1]);
                                    nib4_to_bf16(n1_, o[2], o[3]);
                                } else {
                                    nib4_to_f16(n0_, o[0], o[1]);
                                    nib4_to_f16(n1_, o[2], o[3]);
                                }
                            }
                            if constexpr (F32) bx[0] = as_bf16x8(o);
                            else bf = __builtin_bit_cast(f16x8, make_uint4(o[0], o[1], o[2], o[3]));
                            d = (float)*(const f16*)(sg + L::S_OFF + (mat * 16 * TN + r) * 4 + kk * 2);
                        } else {
                            bf = *(const f16x8*)(bq + r * 128 + ((4 * kk + g) ^ swz_a(r)) * 16);
                            if constexpr (F32) {
                                float wv[8];
#pragma unroll
                                for (int e = 0; e < 8; e++) wv[e] = (float)bf[e];
                                bf16_split(wv, bx);
                            }
                        }
#pragma unroll
                        for (int i = 0; i < TM; i++) {
                            f32x4 c = QUANT || F32 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[mat][i][j];
                            if constexpr (F32) {
                                constexpr int WT = FMT == DT_F16 ? 2 : 1;
#pragma unroll
                                for (int t = WT + 1; t >= 0; t--)  // terms of order t: x's n-th by w's (t - n)-th
#pragma unroll
                                    for (int n = 2; n >= 0; n--)
                                        if (t - n >= 0 && t - n < WT)
                                            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[i][n], bx[t - n], c, 0, 0, 0);
                            } else {
                                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bf, c, 0, 0, 0);
                                if constexpr (TT) c = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], bf, c, 0, 0, 0);
                            }
                            if constexpr (QUANT) acc[mat][i][j] += d * c;
                            else if constexpr (F32) acc[mat][i][j] += c;
                            else acc[mat][i][j] = c;
                        }
                    }
            }
        };
        for (int s = 0; s < min(D, cnt); s++) issue(lds_addr(ring + s * L::BYTES), k0 + s, tt_c);
        if constexpr (NORM) {
            // CPUOps.rmsNorm (CPUOps.swift:144-159), a row per wave in registers
            // as in rmsnorm_rows_kernel (the same operations, so the same bits).
            constexpr int RPW = (16 * TM + NW - 1) / NW;
            const int n4 = K >> 2;
            float4 v[RPW][NV], gv[NV];
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const int i = lane + 64 * k;
                gv[k] = i < n4 ? ((const float4*)p.in.gain)[i] : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < RPW; q++) {
                    const float4* xr = (const float4*)(p.in.xf + (int64_t)min(m0 + wave + q * NW, M - 1) * p.in.ldx);
                    v[q][k] = i < n4 ? xr[i] : float4{0.f, 0.f, 0.f, 0.f};
                }
            }
#pragma unroll
            for (int q = 0; q < RPW; q++) {
                const int row = wave + q * NW;
                if (row >= 16 * TM) break;
                const float scale = rms_scale(v[q], K, p.in.eps);
#pragma unroll
                for (int k = 0; k < NV; k++) {
                    const int i = lane + 64 * k;
                    if (i >= n4) break;
                    const float4 yv = rms_scaled(v[q][k], scale, gv[k]);
                    if constexpr (F32) {
                        *(f32x4*)(rows + row * pitch + 16 * i) = f32x4{yv.x, yv.y, yv.z, yv.w};
                        continue;
                    }
                    const f16x4 hi = f16_first(yv);
                    *(f16x4*)(rows + row * pitch + 8 * i) = hi;
                    if constexpr (TT) *(f16x4*)(rows + (16 * TM + row) * pitch + 8 * i) = f16_second(yv, hi);
                }
            }
            __syncthreads();
        }
        for (int i = 0; i < cnt; i++) {
            // stage i has landed (the D - 1 after it stay in flight, or near the
            // end none is left out of the wait); only this wave reads it
            if (i + D <= cnt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * PER) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            uint8_t* const slot = ring + (i % D) * L::BYTES;
            compute(slot, k0 + i);
            if (i + D < cnt) {
                // the reads of this slot have returned before the DMA overwrites it
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                issue(lds_addr(slot), k0 + i + D, tt_c);
            }
        }
    };
    if constexpr (F32) {
        run(std::false_type{});
    } else {
        if (use_lo) run(std::true_type{});
        else run(std::false_type{});
    }

    // No DMA may still be writing LDS, and every wave is done reading it.
    wait_stage_barrier<0>();
    f32x4* const red = (f32x4*)smem;  // [NW][NB * F][64]
#pragma unroll
    for (int mat = 0; mat < NB; mat++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) red[(wave * NB * F + mat * F + i * TN + j) * 64 + lane] = acc[mat][i][j];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < FW; k++) {
        const int f = wave + k * NW;
        if (f >= F) break;
        f32x4 s[NB];
#pragma unroll
        for (int mat = 0; mat < NB; mat++) {
            s[mat] = red[(mat * F + f) * 64 + lane];
#pragma unroll
            for (int v = 1; v < NW; v++) s[mat] += red[(v * NB * F + mat * F + f) * 64 + lane];
        }
        // C layout of the 16x16 MFMA: lane holds rows 4*(lane/16)+r, column lane%16
        const int mb = m0 + 16 * (f / TN) + 4 * g, g0 = n0 + 16 * (f % TN), n = g0 + l16;
        if constexpr (MODE == GEMM_QKV_ROPE) {
#pragma clang fp contract(off)
            // As in qkv_rope_epilogue (kernels_gemm.hip): a fragment never
            // straddles a head; the RoPE partner is the neighbouring lane.
            const QkvRope& o = p.qkv;
            const int QW = o.heads * o.hd, KW = o.kv_heads * o.hd;
            if (g0 >= N) break;  // N % 16 == 0: whole fragments
            const int region = g0 < QW ? 0 : g0 < QW + KW ? 1 : 2;
            const int cn = n - (region == 0 ? 0 : region == 1 ? QW : QW + KW);
            const bool odd = lane & 1;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = mb + r;
                float out = s[0][r];
                const float pv = dpp_mov<0xB1>(out);  // every lane, before the edge test
                if (region != 2) {
                    const float t1 = out * pre[k][r][0], t2 = pv * (odd ? pre[k][r][1] : -pre[k][r][1]);
                    out = t1 + t2;
                }
                if (m >= M) continue;
                const f16 ho = (f16)out;
                if (region == 0) {
                    const int64_t at = (int64_t)m * p.ldy + n;
                    if constexpr (F32) {
                        p.y[at] = out;
                    } else {
                        p.yh[at] = ho;
                        if (p.yhlo && m >= p.lo_out_row0) p.yhlo[at] = (f16)(out - (float)ho);
                    }
                } else {
                    f16* c = region == 1 ? o.kc : o.vc;
                    c[((int64_t)(cn / o.hd) * o.capacity + o.pos + m) * o.hd + cn % o.hd] = ho;
                }
            }
        } else {
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = mb + r;
                if (m >= M) continue;
                const int64_t at = (int64_t)m * p.ldy + n;
                if constexpr (MODE == GEMM_STORE) {
                    p.y[at] = s[0][r];
                } else if constexpr (MODE == GEMM_ACC) {
                    p.y[at] = pre[k][r][0] + s[0][r];
                } else {
                    const float gt = s[0][r];
                    if constexpr (F32) {
                        p.y[at] = (gt / (1.0f + expf(-gt))) * s[NB - 1][r];
                    } else {
                        const float v = (gt / (1.0f + __expf(-gt))) * s[NB - 1][r];
                        const f16 hv = (f16)v;
                        p.yh[at] = hv;
                        if (p.yhlo && m >= p.lo_out_row0) p.yhlo[at] = (f16)(v - (float)hv);
                    }
                }
            }
        }
    }
}

template <int FMT, int MODE, int TM, int TN, int NW, int D, int NV, bool F32>
hipError_t run_small(const SmallArgs& a, hipStream_t st) {
    const int tiles = ((a.M + 16 * TM - 1) / (16 * TM)) * ((a.w.rows + 16 * TN - 1) / (16 * TN));
    const size_t lds = small_lds<FMT, MODE, TM, TN, NW, D, NV, F32>(a.w.cols);
    auto* kernel = small_gemm_kernel<FMT, MODE, TM, TN, NW, D, NV, F32>;
    static OncePerDevice once;
    if (hipError_t e = allow_whole_lds(once, (const void*)kernel)) return e;
    kernel<<<tiles, 64 * NW, lds, st>>>(a);
    return hipGetLastError();
}

// Tile families, smallest first.  F16 weight stages are twice the size, and
// SwiGLU keeps two of them: the largest tile's then leave room for four waves.
// Normalised rows and float32 ones take the two smallest.
template <int FMT, int MODE, int NV, bool F32>
hipError_t run_family(int family, const SmallArgs& a, hipStream_t st) {
    constexpr int DW = FMT == DT_F16 && MODE == GEMM_SWIGLU ? 1 : 2;
    switch (family) {
    case 0: return run_small<FMT, MODE, 1, 1, 8, 2, NV, F32>(a, st);
    case 1: return run_small<FMT, MODE, 1, 2, 8, DW, NV, F32>(a, st);
    case 2:
        if constexpr (NV == 0 && !F32) return run_small<FMT, MODE, 2, 2, 8, 1, 0, false>(a, st);
        break;
    case 3:
        if constexpr (NV == 0 && !F32) return run_small<FMT, MODE, 2, 4, DW == 1 ? 4 : 8, 1, 0, false>(a, st);
        break;
    }
    return hipErrorNotSupported;
}

template <int FMT, int NV, bool F32>
hipError_t run_mode(int mode, int family, const SmallArgs& a, hipStream_t st) {
    switch (mode) {
    case GEMM_STORE: return run_family<FMT, GEMM_STORE, NV, F32>(family, a, st);
    case GEMM_SWIGLU: return run_family<FMT, GEMM_SWIGLU, NV, F32>(family, a, st);
    case GEMM_QKV_ROPE: return run_family<FMT, GEMM_QKV_ROPE, NV, F32>(family, a, st);
    case GEMM_ACC:
        if constexpr (NV == 0) return run_family<FMT, GEMM_ACC, 0, F32>(family, a, st);
        break;
    }
    return hipErrorNotSupported;
}

template <int FMT>
hipError_t run_input(int mode, int family, const SmallArgs& a, hipStream_t st) {
    const bool norm = a.in.gain != nullptr;
    if (a.in.f32)
        return norm ? run_mode<FMT, kNormV, true>(mode, family, a, st) : run_mode<FMT, 0, true>(mode, family, a, st);
    return norm ? run_mode<FMT, kNormV, false>(mode, family, a, st) : run_mode<FMT, 0, false>(mode, family, a, st);
}

}  // namespace

// The rule: the smallest tile whose grid is at most one workgroup per CU, or
// none (the pipelined tiles of kernels_gemm.hip, which share operands better,
// take the grids past that).  Every family costs about a launch, one memory
// round trip and its tile's bytes, so the smallest wins while each CU runs one.
// A second workgroup on some CUs takes most of that again: past the line the
// 32x64 tiles lose up to 22% or, where K is long and the pipelined tiles pay its
// length in stages, gain up to 8% (the bracketed figures), so the line stays at
// the last grid that always gains.  Two activation terms, Q8_0,
// weights from HBM, us per launch (pipelined tiles -> these):
//   135M shape     QKV          gate+up       down         Wo
//    11 rows    7.8 -> 3.6   10.0 -> 3.7   11.7 -> 3.9   6.7 -> 3.3
//    64 rows    8.3 -> 3.8   10.8 -> 4.5   11.6 -> 4.0   6.5 -> 3.3
//   256 rows    8.5 -> 5.1   11.2 -> 7.9   11.8 -> 6.0   6.5 -> 4.5
//   512 rows    8.6 -> 6.1   11.4 (13.9)   12.2 -> 7.7   6.8 -> 5.3
//   1.7B shape
//    11 rows   16.5 -> 6.2   28.8 -> 10.0  49.4 -> 9.3  15.0 -> 4.2
//    64 rows   16.9 -> 12.4  29.0 -> 18.5  50.0 -> 13.4 14.8 -> 5.5
//   300 rows   26.9 (31.4)   56.9 (61.6)   51.3 (47.2)  15.5 (15.2)
// (figures in brackets: these tiles past one workgroup per CU, not taken).
// With the RMSNorm in the kernel (the two smallest tiles, K <= 1,024), norm
// kernel + GEMM -> one launch: 135M QKV at 64 rows 2.6 + 3.8 -> 5.2 us, gate+up
// at 11 rows 2.6 + 3.7 -> 5.3; on the 32-row tiles it gained nothing (256 rows
// 2.5 + 4.9 -> 7.5), and at K = 2,048 the rows leave no room for the ring
// (2.8 + 6.2 -> 11.2).
// From 768 rows on, the length of the shortest half of a prompt split over two
// streams, the pipelined tiles keep every shape: they sum K in one order
// whatever the tile, so a split prompt's one-term rows are those of an unsplit
// one.
// Float32 rows (fewer than 16) have no pipelined form: the 16x32 tiles take the
// larger grids too.
static int small_family(int m, const DevMatrix& w, const SmallGemmInput& in) {
    static const int tile[4][2] = {{16, 16}, {16, 32}, {32, 32}, {32, 64}};
    const int64_t cus = device_cus();
    auto fits = [&](int f) {
        return (int64_t)((m + tile[f][0] - 1) / tile[f][0]) * ((w.rows + tile[f][1] - 1) / tile[f][1]) <= cus;
    };
    if (in.f32) return fits(0) ? 0 : 1;
    const char* forced = std::getenv("ALPACA_HIP_GEMM_TILE");  // a pipelined tile, or none (tuning and tests)
    if (m >= 768 || (forced && *forced)) return -1;
    for (int f = 0; f < (in.gain ? 2 : 4); f++)
        if (fits(f)) return f;
    return -1;
}

bool gemm_small_takes(const SmallGemmInput& in, int m, const DevMatrix& w, const DevMatrix* w_up) {
    const bool norm = in.gain != nullptr, quant = w.dtype != DT_F16;
    // 64-wide stages, 16-byte aligned rows, the stage-major scales, and operands
    // that 32-bit byte offsets reach
    if (w.cols % SK || in.ldx % 8 || (quant && (!w.s2 || (w_up && !w_up->s2)))) return false;
    if ((int64_t)w.rows * w.cols * 2 > INT32_MAX || (int64_t)m * in.ldx * 4 > INT32_MAX) return false;
    if (norm && (w.cols > 256 * kNormV || ((uintptr_t)in.gain & 15))) return false;
    if (norm || in.f32 ? ((uintptr_t)in.xf & 15) != 0 : (((uintptr_t)in.x | (uintptr_t)in.xlo) & 15) != 0) return false;
    return small_family(m, w, in) >= 0;
}

hipError_t launch_gemm_small(const SmallGemmInput& in, int m, const DevMatrix& w, const DevMatrix* w_up, float* y,
                             f16* yh, f16* yhlo, int ldy, int mode, const QkvRope* rope, hipStream_t st, int lo_row0,
                             int lo_out_row0, int lo_col0) {
    if (m <= 0) return hipSuccess;
    if (!gemm_small_takes(in, m, w, w_up)) return hipErrorNotSupported;
    if (mode == GEMM_QKV_ROPE &&
        (!rope || rope->hd % 16 || w.rows != (rope->heads + 2 * rope->kv_heads) * rope->hd))
        return hipErrorInvalidValue;  // a fragment must not straddle a head
    const int family = small_family(m, w, in);
    SmallArgs a;
    a.in = in;
    a.M = m;
    a.w = w;
    a.u = w_up ? *w_up : w;
    a.y = y;
    a.yh = yh;
    a.yhlo = yhlo;
    a.ldy = ldy;
    a.lo_row0 = lo_row0;
    a.lo_out_row0 = lo_out_row0;
    a.lo_col0 = lo_col0;
    if (rope) a.qkv = *rope;
    // An XCD's tiles share weights (column by column) or activations (row by
    // row), whichever are more bytes.
    const int64_t wb = (int64_t)w.rows * (w.dtype == DT_Q8_0 ? 34 : w.dtype == DT_Q4_0 ? 18 : 64) * (w_up ? 2 : 1);
    a.by_cols = wb >= (int64_t)m * 128;
    switch (w.dtype) {
    case DT_Q8_0: return run_input<DT_Q8_0>(mode, family, a, st);
    case DT_Q4_0: return run_input<DT_Q4_0>(mode, family, a, st);
    default: return run_input<DT_F16>(mode, family, a, st);
    }
}
