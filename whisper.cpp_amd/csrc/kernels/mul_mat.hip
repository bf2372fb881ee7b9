// MUL_MAT for gfx950 (ggml_compute_forward_mul_mat, ggml/src/ggml-cpu/ggml-cpu.c:1266-1458):
//   dst[m, n] = sum_k src0[k, m] * src1[k, n]        src0 = "W" (weights, rows m), src1 = "X" (rows n)
//
// This file: the tiled MFMA GEMM (many columns; f16 operands, f32 accumulation, whatever the weights' type: one pass brings
// blocks to f16), k_mul_mat_generic for what no other kernel takes, and the dispatch.  The quantized few-column products are
// in gemv.hip, the split-K products over f16 weights in gemm_ks.hip.
#include "common.h"

#include <algorithm>
#include <atomic>
#include <mutex>
#include <stdlib.h>
#include <type_traits>


// ------------------------------------------------------------------------------------------------------
// shared: epilogue
// ------------------------------------------------------------------------------------------------------

#include "mul_mat_args.h"
#include "gemm_ks.h"
#include "gemv.h"

// The same for the 16 registers of one 32x32 accumulator patch (column m, rows n[0..15]) and the stores.  All loads of
// one kind are issued together before their first use; rows beyond N and columns beyond M are computed from clamped
// addresses and not stored.
// The part of the GELU table that the values in front of a GELU fall into, as a workgroup keeps it in LDS: the f16 patterns
// of |x| < 8 — 0x0000 .. 0x47ff and 0x8000 .. 0xc7ff, 2 x 18432 entries, 73728 bytes — positive half first.
#define GELU_LDS_HALF  0x4800
#define GELU_LDS_BYTES (2 * GELU_LDS_HALF * 2)

// FULL: the whole tile lies inside dst (no row or column of the patch is clamped or masked)
template <bool FULL>
__device__ __forceinline__ void patch_epilogue(float16_t v, const epi_args & e, char * db, int64_t batch_off, int64_t d_nb1,
                                               int64_t m, int64_t M, const int64_t (&n)[16], int64_t N, const uint16_t * gelu_lds = nullptr) {
    const bool    m_ok = FULL || m < M;
    const int64_t mc   = m_ok ? m : M - 1;
    int64_t nc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) nc[i] = FULL || n[i] < N ? n[i] : N - 1;
    if (e.flags & MI355X_EPI_BIAS) {
        const float b = e.bias[mc];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] += b;
    }
    if (e.flags & MI355X_EPI_BIAS_COL) {
        float b[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) b[i] = e.bias[nc[i]];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] += b[i];
    }
    if (e.flags & MI355X_EPI_GELU) {
        if (gelu_lds) {
            // 64 gathers per lane out of the 128 KB table in global memory cost the FFN-up product 10 us of its 45; out of
            // LDS, 8.  A value near 8 or more in magnitude (none in a whisper model's activations) sends the wavefront through
            // the general form: the clamps at +-10 and the table in global memory for what the slice does not hold.
            bool far = false;
#pragma unroll
            for (int i = 0; i < 16; ++i) far = far || !(fabsf(v[i]) < 7.99f);   // (f16 rounds up to 8 from 7.998; NaN is far)
            if (!__any(far)) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t hb = f2h_bits(v[i]);
                    v[i] = h2f(gelu_lds[(hb & 0x7FFFu) + (hb >> 15) * GELU_LDS_HALF]);
                }
            } else {
                uint32_t hb[16]; uint16_t t[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    hb[i] = f2h_bits(v[i]);
                    const uint32_t a = hb[i] & 0x7FFFu;
                    t[i] = gelu_lds[(a < GELU_LDS_HALF ? a : 0u) + (hb[i] >> 15) * GELU_LDS_HALF];
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) if ((hb[i] & 0x7FFFu) >= GELU_LDS_HALF) t[i] = e.gelu[hb[i]];
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = v[i] <= -10.0f ? 0.0f : v[i] >= 10.0f ? v[i] : h2f(t[i]);
            }
        } else {
            uint16_t t[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) t[i] = e.gelu[f2h_bits(v[i])];
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = v[i] <= -10.0f ? 0.0f : v[i] >= 10.0f ? v[i] : h2f(t[i]);
        }
    }
    if (e.flags & MI355X_EPI_SCALE) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] *= e.scale;
    }
    if (e.flags & MI355X_EPI_RESIDUAL) {
        float r[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) r[i] = *(const float *)(e.residual + batch_off + nc[i] * d_nb1 + mc * 4);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] += r[i];
    }
    if (e.flags & MI355X_EPI_OUT_F16) {
#pragma unroll
        for (int i = 0; i < 16; ++i) if (m_ok && (FULL || n[i] < N)) *(half_t *)(db + n[i] * d_nb1 + m * 2) = (half_t) v[i];
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) if (m_ok && (FULL || n[i] < N)) *(float *)(db + n[i] * d_nb1 + m * 4) = v[i];
    }
}

// The same for a patch formed the other way round (the weights as the matrix instruction's A operand): the lane owns ONE dst row
// n and 16 of the 32 consecutive m of a patch row — m = mb + 8 q + t, q = e / 4, t = e % 4, with mb = the patch's first m +
// 4 (lane / 32) — and lane + 32 owns the other 16.  That is half a Q8_0 block per lane: the block maximum is 8 three-operand
// maxima and one exchange with lane + 32, both divisions are the lane's own, bias, residual and stores move four consecutive
// values at a time.  MI355X_EPI_EMIT_F16: the image f16(q * d) of the patch, as the src1 conversion pass of the product that reads
// dst next would make it, goes to `stage` (LDS; half4 q of this lane at 16 q).
// M a multiple of 32 (a patch lies inside dst's columns or outside); FULL: the patch is inside and n < N.
template <bool FULL>
__device__ __forceinline__ void patch_epilogue_t(float16_t v, const epi_args & e, char * db, int64_t batch_off, int64_t d_nb1,
                                                 int64_t mb, int64_t M, int64_t n, int64_t N, const uint16_t * gelu_lds, char * stage) {
    const bool    ok = FULL || (n < N && mb < M);
    const int64_t nc = FULL || n < N ? n : N - 1;
    const int64_t mc = FULL || mb < M ? mb : M - 32 + (mb & 31);
    if (e.flags & MI355X_EPI_BIAS) {
        float4 b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = *(const float4 *)(e.bias + mc + 8 * q);
#pragma unroll
        for (int q = 0; q < 4; ++q) { v[4 * q] += b[q].x; v[4 * q + 1] += b[q].y; v[4 * q + 2] += b[q].z; v[4 * q + 3] += b[q].w; }
    }
    if (e.flags & MI355X_EPI_BIAS_COL) {
        const float b = e.bias[nc];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] += b;
    }
    if (e.flags & MI355X_EPI_GELU) {
        if (gelu_lds) {
            // the table slice in LDS holds |x| < 8: the f16 patterns below 0x4800 (infinity and NaN lie above); one integer
            // maximum over the patterns decides for the wavefront, the general form is the one of patch_epilogue
            uint32_t hb[16], top = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i) { hb[i] = f2h_bits(v[i]); top = max(top, hb[i] & 0x7FFFu); }
            if (!__any(top >= GELU_LDS_HALF)) {
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = h2f(gelu_lds[(hb[i] & 0x7FFFu) + (hb[i] >> 15) * GELU_LDS_HALF]);
            } else {
                uint16_t t[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t a = hb[i] & 0x7FFFu;
                    t[i] = gelu_lds[(a < GELU_LDS_HALF ? a : 0u) + (hb[i] >> 15) * GELU_LDS_HALF];
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) if ((hb[i] & 0x7FFFu) >= GELU_LDS_HALF) t[i] = e.gelu[hb[i]];
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = v[i] <= -10.0f ? 0.0f : v[i] >= 10.0f ? v[i] : h2f(t[i]);
            }
        } else {
            uint16_t t[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) t[i] = e.gelu[f2h_bits(v[i])];
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = v[i] <= -10.0f ? 0.0f : v[i] >= 10.0f ? v[i] : h2f(t[i]);
        }
    }
    if (e.flags & MI355X_EPI_SCALE) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] *= e.scale;
    }
    if (e.flags & MI355X_EPI_RESIDUAL) {
        float4 r[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] = *(const float4 *)(e.residual + batch_off + nc * d_nb1 + (mc + 8 * q) * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) { v[4 * q] += r[q].x; v[4 * q + 1] += r[q].y; v[4 * q + 2] += r[q].z; v[4 * q + 3] += r[q].w; }
    }
    if (e.flags & MI355X_EPI_OUT_F16) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (ok) *(half4_t *)(db + n * d_nb1 + (mb + 8 * q) * 2) = (half4_t){ (half_t) v[4 * q], (half_t) v[4 * q + 1], (half_t) v[4 * q + 2], (half_t) v[4 * q + 3] };
    } else if (!(e.flags & MI355X_EPI_IMAGE_ONLY)) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (ok) *(float4 *)(db + n * d_nb1 + (mb + 8 * q) * 4) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
    }
    // the image: rounded to Q8_0 as the product that reads dst next rounds its rows (quantize_row_q8_0, then widened)
    float amax = fmaxf(fabsf(v[0]), fabsf(v[1]));
#pragma unroll
    for (int i = 2; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
    {   // ... and the half of the block that lane ^ 32 holds (v_permlane32_swap of the value with itself: own half, other half)
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(amax), __float_as_uint(amax), false, false);
        amax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
    const float dq = h2f(f2h_bits(div127(amax)));
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        // (the addend +0 of the multiply-add turns a product -0 into the +0 that an integer quant of zero gives)
        const half4_t h = { (half_t) __builtin_fmaf(rintf(v[4 * q] * id), dq, 0.0f), (half_t) __builtin_fmaf(rintf(v[4 * q + 1] * id), dq, 0.0f),
                            (half_t) __builtin_fmaf(rintf(v[4 * q + 2] * id), dq, 0.0f), (half_t) __builtin_fmaf(rintf(v[4 * q + 3] * id), dq, 0.0f) };
        *(half4_t *)(stage + 16 * q) = h;
    }
}


// ------------------------------------------------------------------------------------------------------
// block -> 32 f16 weights
// ------------------------------------------------------------------------------------------------------

// bytes (b0,b1) / (b2,b3) of v, each in [0,255], become the f16 pair (b - bias): 0x6400|b is the f16 1024+b.
__device__ __forceinline__ half2_t bytes_lo_to_half2(uint32_t v, half2_t bias) {
    uint32_t u = (v & 0xFFu) | ((v << 8) & 0xFF0000u) | 0x64006400u;
    half2_t h; __builtin_memcpy(&h, &u, 4);
    return h - bias;
}
__device__ __forceinline__ half2_t bytes_hi_to_half2(uint32_t v, half2_t bias) {
    uint32_t u = ((v >> 16) & 0xFFu) | ((v >> 8) & 0xFF0000u) | 0x64006400u;
    half2_t h; __builtin_memcpy(&h, &u, 4);
    return h - bias;
}

// f16(d * q) equals the f16 rounding of the exact product: q is a small integer, so (q as f16) * (d as f16)
// in one v_pk_mul_f16 rounds once.
__device__ __forceinline__ void q5_0_to_half32(uint32_t d_bits, uint32_t qh, const uint32_t qs[4], half8_t out[4]) {
    half_t d; { uint16_t t = (uint16_t) d_bits; __builtin_memcpy(&d, &t, 2); }
    const half2_t d2 = { d, d };
    const half2_t bias = { (half_t) 1040.0f, (half_t) 1040.0f };   // 1024 + 16
    half2_t * o = (half2_t *) out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t q  = qs[i];
        const uint32_t lo = (q & 0x0F0F0F0Fu)        | spread4_to_bit4((qh >> (4*i))      & 0xFu);
        const uint32_t hi = ((q >> 4) & 0x0F0F0F0Fu) | spread4_to_bit4((qh >> (16 + 4*i)) & 0xFu);
        o[2*i + 0]     = bytes_lo_to_half2(lo, bias) * d2;   // k = 4i, 4i+1
        o[2*i + 1]     = bytes_hi_to_half2(lo, bias) * d2;   // k = 4i+2, 4i+3
        o[8 + 2*i + 0] = bytes_lo_to_half2(hi, bias) * d2;   // k = 16+4i ..
        o[8 + 2*i + 1] = bytes_hi_to_half2(hi, bias) * d2;
    }
}
__device__ __forceinline__ void q8_0_to_half32(uint32_t d_bits, const uint32_t qs[8], half8_t out[4]) {
    half_t d; { uint16_t t = (uint16_t) d_bits; __builtin_memcpy(&d, &t, 2); }
    const half2_t d2 = { d, d };
    const half2_t bias = { (half_t) 1152.0f, (half_t) 1152.0f };   // 1024 + 128
    half2_t * o = (half2_t *) out;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t v = qs[i] ^ 0x80808080u;                    // int8 -> biased uint8
        o[2*i + 0] = bytes_lo_to_half2(v, bias) * d2;
        o[2*i + 1] = bytes_hi_to_half2(v, bias) * d2;
    }
}

// ------------------------------------------------------------------------------------------------------
// MFMA GEMM: operand conversion passes + one f16 x f16 -> f32 kernel
//
// Both operands reach the matrix cores as dense f16 rows [rows][K]:
//   * src1 (F32) is converted by k_x_to_f16.  For quantized weights the CPU backend first rounds src1 to Q8_0
//     (ggml-cpu.c:1328-1363, quantize_row_q8_0 ggml-cpu-quants.c:808-865): the pass reproduces that rounding —
//     block amax, id = 127/amax, round half to even, d stored as f16 — and writes f16(q * d).  For F16 / F32
//     weights (or when the caller asks for un-rounded activations) it is a plain f32 -> f16 conversion, which is
//     what the CPU backend does for F16 weights.
//   * src0 blocks are expanded by k_w_to_f16 to f16(d * q) unless src0 already is F16.  A caller that multiplies by
//     the same weights many times keeps that f16 image itself and passes it as an F16 src0 with MI355X_MM_ACT_Q8_0.
// ------------------------------------------------------------------------------------------------------


// one thread per 32 weights
template <int T0>
__global__ void k_w_to_f16(const char * __restrict__ w, half_t * __restrict__ out, int64_t K, int64_t M, int64_t w_nb1, int64_t w_nb2,
                           int64_t ne02, int64_t w_nb3, int64_t slice_halves) {
    const int64_t t   = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nbk = K / QK;
    if (t >= nbk * M) return;
    const int64_t m = t / nbk, kb = t % nbk, b = blockIdx.y;
    const uint8_t * row = (const uint8_t *) w + m * w_nb1 + (b % ne02) * w_nb2 + (b / ne02) * w_nb3;
    half8_t o[4];
    if constexpr (T0 == MI355X_TYPE_Q5_0) {
        const uint8_t * p = row + kb * 22;
        const u128a2 q = *(const u128a2 *)(p + 6);
        const uint32_t qs[4] = { q.x, q.y, q.z, q.w };
        q5_0_to_half32(*(const uint16_t *) p, *(const u32a2 *)(p + 2), qs, o);
    } else if constexpr (T0 == MI355X_TYPE_Q8_0) {
        const uint8_t * p = row + kb * 34;
        const u128a2 q0 = *(const u128a2 *)(p + 2), q1 = *(const u128a2 *)(p + 18);
        const uint32_t qs[8] = { q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w };
        q8_0_to_half32(*(const uint16_t *) p, qs, o);
    } else {
        const float4 * p = (const float4 *)(row + kb * QK * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 u = p[2*i], v = p[2*i + 1];
            o[i] = (half8_t){ (half_t) u.x, (half_t) u.y, (half_t) u.z, (half_t) u.w, (half_t) v.x, (half_t) v.y, (half_t) v.z, (half_t) v.w };
        }
    }
    half8_t * dst = (half8_t *)(out + b * slice_halves + m * K + kb * QK);
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[i] = o[i];
}

// 8 lanes per 32 values, 4 each
template <bool Q8>
__global__ void k_x_to_f16(const char * __restrict__ x, half_t * __restrict__ out, int64_t K, int64_t N,
                           int64_t x_nb1, int64_t x_nb2, int64_t ne12, int64_t x_nb3, int64_t slice_halves) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x, k4 = (uint32_t)(K / 4);         // (k4 N < 2^32: a batch slice of 2^34 values is no case)
    const int64_t b = blockIdx.y;
    if (t >= k4 * (uint32_t) N) return;                                     // whole 8-lane groups leave together (K % 32 == 0 when Q8)
    const uint32_t n = t / k4, c = t - n * k4, b3 = div_count(blockIdx.y, ne12), b2 = blockIdx.y - b3 * (uint32_t) ne12;
    const float4 v = *(const float4 *)(x + n * x_nb1 + b2 * x_nb2 + b3 * x_nb3 + c * 16);
    half4_t h;
    if (Q8) {
        float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
        amax = lanes_max<8>(amax);
        const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
        const float d  = h2f(f2h_bits(div127(amax)));                      // the scale goes through f16, like block_q8_0.d
        // (+ 0.0f: a quant that rounds to -0 is the integer 0, whose product with d is +0)
        h = (half4_t){ (half_t)((rintf(v.x * id) + 0.0f) * d), (half_t)((rintf(v.y * id) + 0.0f) * d), (half_t)((rintf(v.z * id) + 0.0f) * d), (half_t)((rintf(v.w * id) + 0.0f) * d) };
    } else {
        h = (half4_t){ (half_t) v.x, (half_t) v.y, (half_t) v.z, (half_t) v.w };
    }
    *(half4_t *)(out + b * slice_halves + n * K + c * 4) = h;
}

// f16 x f16 -> f32 GEMM.  256 threads = 4 wavefronts in a 2 x 2 grid; a wavefront owns TI x TJ accumulator patches of
// 32 (src1 rows, n) x 32 (weight rows, m), each a v_mfma_f32_32x32x16_f16 chain.  src1 rows are the MFMA A operand and
// weight rows the B operand, so a lane's accumulator column is an m index and every store instruction writes 32
// consecutive values of a dst row.  K advances 64 at a time through two LDS buffers: while the matrix cores work on
// step s, the global loads of step s+2 are in flight and step s+1 moves from registers to the other buffer, with one
// barrier per step.  LDS rows are padded to 144 B so that the 16-byte operand reads of 16 consecutive rows hit
// distinct banks.  What bounds the kernel is the staging, not the K loop: with the operands already in LDS the loop runs
// at 1400 TFLOP/s (8192^3); the LDS stores bring that to 1155 and the global loads to 805 — a 128 x 128 x 64 step
// fetches 32 KB through a vector memory path of 64 B per clock and CU, as many clocks as its matrix instructions take.
#define GB_K  64
#define GB_LD (GB_K + 8)


// What follows the K loop of a tile: GELU reads its table from LDS when the operand buffers, free now (the loop's last barrier
// is behind every wavefront), are large enough to hold the part that matters (TABLE_FITS); then the 32x32 patches.
// NT: threads of the workgroup (more than a BN x BM tile has patches for: the patches belong to the first 256).  EMIT: the patches
// were formed with the weights as the matrix instruction's A operand — lanes own dst rows, registers own columns.  table_there: the
// GELU slice is in LDS already.
template <int TI, int TJ, bool EMIT, bool TABLE_FITS, int NT = 256, int BN = 64 * TI, int BM = 64 * TJ>
__device__ __forceinline__ void gemm_tile_epilogue(float16_t (&acc)[TI][TJ], const mm_args & a, const epi_args & epi, char * db, int64_t batch_off, int64_t d_nb1,
                                                   int64_t n0, int64_t m0, int wn, int wmo, char * smem, bool table_there = false) {
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const uint16_t * gelu_lds = nullptr;
    if constexpr (TABLE_FITS) {
        if (table_there) gelu_lds = (const uint16_t *) smem;
        else if (epi.flags & MI355X_EPI_GELU) {
            const u32x4 * pos = (const u32x4 *) epi.gelu, * neg = (const u32x4 *)(epi.gelu + 0x8000);
            u32x4 * dst = (u32x4 *) smem;
            constexpr int pieces = GELU_LDS_HALF * 2 / 16;
            for (int p = tid; p < pieces; p += NT) { dst[p] = pos[p]; dst[pieces + p] = neg[p]; }
            __syncthreads();
            gelu_lds = (const uint16_t *) smem;
        }
    }
    if (NT > 256 && BN * BM == 64 * TI * 64 * TJ && tid >= 256) return;
    if constexpr (EMIT) {
        // accumulator register e of a 32x32 patch: column (= n) lane%32, row (= m) 8*(e/4) + 4*g + e%4
        // The image leaves through LDS: a lane's half4s go to 32 different rows, 8 bytes each, and 32 cache lines to a store made the
        // epilogue longer than the K loop; out of LDS a store is whole 64- or 128-byte row pieces.
        constexpr int PITCH = 64 * TJ + 16;             // bytes of a row of the wavefront's 32 TI x 32 TJ values
        char * stage = smem + (TABLE_FITS ? GELU_LDS_BYTES : 0) + (tid >> 6) * (32 * TI * PITCH);
        auto patches_t = [&](auto full) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    patch_epilogue_t<decltype(full)::value>(acc[i][j], epi, db, batch_off, d_nb1, m0 + wmo + 32 * j + 4 * g, a.M, n0 + wn + 32 * i + l32, a.N, gelu_lds,
                                                            stage + (32 * i + l32) * PITCH + 64 * j + 8 * g);
        };
        if (n0 + BN <= a.N && m0 + BM <= a.M) patches_t(std::true_type{}); else patches_t(std::false_type{});
        constexpr int CPR = 4 * TJ, RPI = 64 / CPR;     // 16-byte chunks of a row; rows of a store
#pragma unroll
        for (int k = 0; k < 32 * TI / RPI; ++k) {
            const int r = k * RPI + lane / CPR, c = lane % CPR;
            const half8_t h = *(const half8_t *)(stage + r * PITCH + c * 16);
            const int64_t n = n0 + wn + r, m = m0 + wmo + 8 * c;
            if (n < a.N && m < a.M) *(half8_t *)(epi.image + n * a.M + m) = h;
        }
        return;
    }
    // accumulator register e of a 32x32 patch: row (= n) 8*(e/4) + 4*g + e%4, column (= m) lane%32
    auto patches = [&](auto full) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            int64_t n[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) n[e] = n0 + wn + 32 * i + 8 * (e >> 2) + 4 * g + (e & 3);
#pragma unroll
            for (int j = 0; j < TJ; ++j)
                patch_epilogue<decltype(full)::value>(acc[i][j], epi, db, batch_off, d_nb1, m0 + wmo + 32 * j + l32, a.M, n, a.N, gelu_lds);
        }
    };
    // tiles inside dst (all but the last row of tiles when N = 1500) store without per-element bounds
    if (n0 + BN <= a.N && m0 + BM <= a.M) patches(std::true_type{}); else patches(std::false_type{});
}

// The loop with the operands on their way through registers: any K that is a multiple of 8.
template <int TI, int TJ>
__device__ __forceinline__ void gemm_f16_tile(const mm_args & a, int tiles_m, int tiles_n, int sw, int tile, const char * wb, const char * xb, char * db,
                                              const epi_args & epi, int64_t batch_off, int64_t d_nb1) {
    constexpr int BN = 64 * TI, BM = 64 * TJ;
    constexpr int XR = BN / 32, WR = BM / 32;          // 16-byte pieces per thread and step
    extern __shared__ __attribute__((aligned(16))) char smem[];
    half_t * xs_base = (half_t *) smem;                // [2][BN * GB_LD]
    half_t * ws_base = xs_base + 2 * BN * GB_LD;       // [2][BM * GB_LD]

    // `tile` counts along a path over the tile grid that walks columns of `sw` m-tiles, each from the first n-panel to the
    // last (m fastest inside the column): a run of consecutive tiles — what one XCD gets, see xcd_run_index — then covers
    // about sqrt(run) tiles in each direction, the shape that touches the fewest X and W rows.
    const int per_col = sw * tiles_n, col = tile / per_col, rem = tile - col * per_col;
    const int cw = min(sw, tiles_m - col * sw);        // (the last column is narrower when sw does not divide tiles_m)
    const int64_t m0 = (int64_t)(col * sw + rem % cw) * BM;
    const int64_t n0 = (int64_t)(rem / cw) * BN;

    const int tid = threadIdx.x;
    const int lc = tid & 7, lr = tid >> 3;             // piece column (8 halves) and first row of this thread
    // rows beyond N / M are read from the last valid row: what they produce is never stored
    const char * xp[XR]; const char * wp[WR];
#pragma unroll
    for (int i = 0; i < XR; ++i) { const int64_t n = n0 + lr + 32 * i; xp[i] = xb + (n < a.N ? n : a.N - 1) * a.x_nb1 + lc * 16; }
#pragma unroll
    for (int i = 0; i < WR; ++i) { const int64_t m = m0 + lr + 32 * i; wp[i] = wb + (m < a.M ? m : a.M - 1) * a.w_nb1 + lc * 16; }

    // two steps of operands are in flight in registers (slot = step % 2); pieces beyond K are read from k = 0 and zeroed
    u32x4 xrs[2][XR], wrs[2][WR];
    auto load = [&](u32x4 (&xr)[XR], u32x4 (&wr)[WR], int64_t k0) __attribute__((always_inline)) {
        const bool kok = k0 + 8 * lc < a.K;
        const int64_t ko = kok ? k0 * 2 : -(int64_t) lc * 16;
#pragma unroll
        for (int i = 0; i < XR; ++i) { const u32x4 v = *(const u32x4 *)(xp[i] + ko); xr[i] = kok ? v : (u32x4){0, 0, 0, 0}; }
#pragma unroll
        for (int i = 0; i < WR; ++i) { const u32x4 v = *(const u32x4 *)(wp[i] + ko); wr[i] = kok ? v : (u32x4){0, 0, 0, 0}; }
    };
    auto store = [&](const u32x4 (&xr)[XR], const u32x4 (&wr)[WR], int buf) __attribute__((always_inline)) {
        half_t * xs = xs_base + buf * BN * GB_LD, * ws = ws_base + buf * BM * GB_LD;
#pragma unroll
        for (int i = 0; i < XR; ++i) *(u32x4 *)(xs + (lr + 32 * i) * GB_LD + 8 * lc) = xr[i];
#pragma unroll
        for (int i = 0; i < WR; ++i) *(u32x4 *)(ws + (lr + 32 * i) * GB_LD + 8 * lc) = wr[i];
    };

    const int lane = tid & 63, wave = tid >> 6;
    const int wn = (wave >> 1) * 32 * TI, wmo = (wave & 1) * 32 * TJ;   // wave patch origin inside the tile
    const int l32 = lane & 31, g = lane >> 5;

    float16_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    const int KT = (int)((a.K + GB_K - 1) / GB_K);
    // one K step: the operand fragments of sub-step kk + 1 are read from LDS while the matrix cores work on kk
    auto mma = [&](int buf) __attribute__((always_inline)) {
        const half_t * xs = xs_base + buf * BN * GB_LD + (wn  + l32) * GB_LD + 8 * g;
        const half_t * ws = ws_base + buf * BM * GB_LD + (wmo + l32) * GB_LD + 8 * g;
        half8_t av[2][TI], bv[2][TJ];
#pragma unroll
        for (int i = 0; i < TI; ++i) av[0][i] = *(const half8_t *)(xs + 32 * i * GB_LD);
#pragma unroll
        for (int j = 0; j < TJ; ++j) bv[0][j] = *(const half8_t *)(ws + 32 * j * GB_LD);
#pragma unroll
        for (int kk = 0; kk < GB_K / 16; ++kk) {
            const int c = kk & 1, nx = c ^ 1;
            if (kk + 1 < GB_K / 16) {
#pragma unroll
                for (int i = 0; i < TI; ++i) av[nx][i] = *(const half8_t *)(xs + 32 * i * GB_LD + (kk + 1) * 16);
#pragma unroll
                for (int j = 0; j < TJ; ++j) bv[nx][j] = *(const half8_t *)(ws + 32 * j * GB_LD + (kk + 1) * 16);
            }
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[c][i], bv[c][j], acc[i][j], 0, 0, 0);
            if (kk + 1 < GB_K / 16) {
                // issue order: one LDS read after each of the first matrix instructions of this sub-step
#pragma unroll
                for (int r = 0; r < TI + TJ; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // 1 MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // 1 DS read
                }
            }
        }
    };
    load(xrs[0], wrs[0], 0);
    if (1 < KT) load(xrs[1], wrs[1], GB_K);
    store(xrs[0], wrs[0], 0);
    if (2 < KT) load(xrs[0], wrs[0], 2 * GB_K);
    __syncthreads();
    auto step = [&](int kt, int buf, u32x4 (&xr)[XR], u32x4 (&wr)[WR]) __attribute__((always_inline)) {   // xr / wr: slot of step kt + 1
        mma(buf);
        if (kt + 1 < KT) {
            store(xr, wr, buf ^ 1);                     // the last readers of that buffer passed the previous barrier
            if (kt + 3 < KT) load(xr, wr, (int64_t)(kt + 3) * GB_K);
        }
        __syncthreads();
    };
    for (int kt0 = 0; kt0 < KT; kt0 += 2) {
        step(kt0 + 0, 0, xrs[1], wrs[1]);
        if (kt0 + 1 < KT) step(kt0 + 1, 1, xrs[0], wrs[0]);
    }

    gemm_tile_epilogue<TI, TJ, false, ((size_t) 2 * (BN + BM) * GB_LD * sizeof(half_t) >= GELU_LDS_BYTES)>(acc, a, epi, db, batch_off, d_nb1, n0, m0, wn, wmo, smem);
}

// The same tile by a workgroup of eight wavefronts in two roles: wavefronts 4 .. 7 move the operands (global loads into a
// register ring, LDS stores of the step after next), wavefronts 0 .. 3 issue the matrix instructions of the current step,
// one barrier per step between them.  In the one-role loop above a wavefront spends two thirds of a step issuing loads and
// stores, during which it issues no matrix instruction; here the matrix wavefronts do nothing else, and a SIMD holds
// one of each role per workgroup.  K a multiple of 64 S.
// NP: threads that move operands (256 or 512), behind the 256 that multiply
template <int TI, int TJ, int S, int NP>
__device__ __forceinline__ void gemm_f16_tile_rs(const mm_args & a, int tiles_m, int tiles_n, int sw, int tile, const char * wb, const char * xb, char * db,
                                                 const epi_args & epi, int64_t batch_off, int64_t d_nb1) {
    constexpr int BN = 64 * TI, BM = 64 * TJ;
    constexpr int RP = NP / 8;                         // rows that the operand threads cover in one pass (8 threads to a row)
    constexpr int XR = BN / RP, WR = BM / RP;          // 16-byte pieces per operand thread and step
    static_assert(BN % RP == 0 && BM % RP == 0, "");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    half_t * xs_base = (half_t *) smem;                // [2][BN * GB_LD]
    half_t * ws_base = xs_base + 2 * BN * GB_LD;       // [2][BM * GB_LD]

    const int per_col = sw * tiles_n, col = tile / per_col, rem = tile - col * per_col;
    const int cw = min(sw, tiles_m - col * sw);
    const int64_t m0 = (int64_t)(col * sw + rem % cw) * BM;
    const int64_t n0 = (int64_t)(rem / cw) * BN;

    const int tid = threadIdx.x;
    const int KT = (int)(a.K / GB_K), last = KT - 1;
    const int lane = tid & 63, wave = (tid >> 6) & 3;
    const int wn = (wave >> 1) * 32 * TI, wmo = (wave & 1) * 32 * TJ;   // (matrix wavefronts) patch origin inside the tile

    float16_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    if (tid >= 256) {
        // ---- operand wavefronts
        const int pt = tid - 256, lc = pt & 7, lr = pt >> 3;
        const char * xp[XR]; const char * wp[WR];
#pragma unroll
        for (int i = 0; i < XR; ++i) { const int64_t n = n0 + lr + RP * i; xp[i] = xb + (n < a.N ? n : a.N - 1) * a.x_nb1 + lc * 16; }
#pragma unroll
        for (int i = 0; i < WR; ++i) { const int64_t m = m0 + lr + RP * i; wp[i] = wb + (m < a.M ? m : a.M - 1) * a.w_nb1 + lc * 16; }
        u32x4 xrs[S][XR], wrs[S][WR];
        auto load = [&](u32x4 (&xr)[XR], u32x4 (&wr)[WR], int64_t k0) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < XR; ++i) xr[i] = *(const u32x4 *)(xp[i] + k0 * 2);
#pragma unroll
            for (int i = 0; i < WR; ++i) wr[i] = *(const u32x4 *)(wp[i] + k0 * 2);
        };
        auto store = [&](const u32x4 (&xr)[XR], const u32x4 (&wr)[WR], int buf) __attribute__((always_inline)) {
            half_t * xs = xs_base + buf * BN * GB_LD, * ws = ws_base + buf * BM * GB_LD;
#pragma unroll
            for (int i = 0; i < XR; ++i) *(u32x4 *)(xs + (lr + RP * i) * GB_LD + 8 * lc) = xr[i];
#pragma unroll
            for (int i = 0; i < WR; ++i) *(u32x4 *)(ws + (lr + RP * i) * GB_LD + 8 * lc) = wr[i];
        };
        // every step loads unconditionally (beyond the end: the last step again), so the waits are counts, not vmcnt(0)
#pragma unroll
        for (int st = 0; st < S; ++st) load(xrs[st], wrs[st], (int64_t) min(st, last) * GB_K);
        store(xrs[0], wrs[0], 0);
        load(xrs[0], wrs[0], (int64_t) min(S, last) * GB_K);
        __syncthreads();                               // step 0 is in LDS
        auto step = [&](int kt, int buf, u32x4 (&xr)[XR], u32x4 (&wr)[WR]) __attribute__((always_inline)) {   // xr / wr: slot of step kt + 1
            store(xr, wr, buf ^ 1);                     // the matrix wavefronts read `buf`; the readers of buf ^ 1 passed the last barrier
            load(xr, wr, (int64_t) min(kt + 1 + S, last) * GB_K);
            __syncthreads();
        };
        for (int kt0 = 0; kt0 < KT; kt0 += S) {
            step(kt0 + 0, 0, xrs[1 % S], wrs[1 % S]);
            step(kt0 + 1, 1, xrs[2 % S], wrs[2 % S]);
            if (S > 2) { step(kt0 + 2, 0, xrs[3 % S], wrs[3 % S]); step(kt0 + 3, 1, xrs[4 % S], wrs[4 % S]); }
        }
    } else {
        // ---- matrix wavefronts
        const int l32 = lane & 31, g = lane >> 5;
        auto mma = [&](int buf) __attribute__((always_inline)) {
            const half_t * xs = xs_base + buf * BN * GB_LD + (wn  + l32) * GB_LD + 8 * g;
            const half_t * ws = ws_base + buf * BM * GB_LD + (wmo + l32) * GB_LD + 8 * g;
            // fragments of sub-step kk + 1 are read while the matrix cores work on kk (two sets of registers: with two
            // workgroups to a CU a wavefront has 128)
            half8_t av[2][TI], bv[2][TJ];
#pragma unroll
            for (int i = 0; i < TI; ++i) av[0][i] = *(const half8_t *)(xs + 32 * i * GB_LD);
#pragma unroll
            for (int j = 0; j < TJ; ++j) bv[0][j] = *(const half8_t *)(ws + 32 * j * GB_LD);
#pragma unroll
            for (int kk = 0; kk < GB_K / 16; ++kk) {
                const int c = kk & 1, nx = c ^ 1;
                if (kk + 1 < GB_K / 16) {
#pragma unroll
                    for (int i = 0; i < TI; ++i) av[nx][i] = *(const half8_t *)(xs + 32 * i * GB_LD + (kk + 1) * 16);
#pragma unroll
                    for (int j = 0; j < TJ; ++j) bv[nx][j] = *(const half8_t *)(ws + 32 * j * GB_LD + (kk + 1) * 16);
                }
#pragma unroll
                for (int i = 0; i < TI; ++i)
#pragma unroll
                    for (int j = 0; j < TJ; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[c][i], bv[c][j], acc[i][j], 0, 0, 0);
                if (kk + 1 < GB_K / 16) {
#pragma unroll
                    for (int r = 0; r < TI + TJ; ++r) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // 1 MFMA
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // 1 DS read
                    }
                }
            }
        };
        __syncthreads();                               // step 0 is in LDS
        for (int kt = 0; kt < KT; kt += 2) {            // (KT is even)
            mma(0); __syncthreads();
            mma(1); __syncthreads();
        }
    }
    // all eight wavefronts are behind the last barrier: the operand buffers are free
    gemm_tile_epilogue<TI, TJ, false, ((size_t) 2 * (BN + BM) * GB_LD * sizeof(half_t) >= GELU_LDS_BYTES), 256 + NP>(acc, a, epi, db, batch_off, d_nb1, n0, m0, wn, wmo, smem);
}

// The same tile with the operands going from global memory straight into LDS (global_load_lds_dwordx4: lane l's 16 bytes
// land at the wave's LDS base + 16 l, no register and no LDS store instruction in between): a step is a wait, a barrier, the
// issue of the loads NBUF - 1 steps ahead and the matrix phase of WN x WM wavefronts, 32 TI x 32 TJ results each.
// What bounds it: a CU takes about 55 KB/us in from L2 (25 B per clock: 14 TB/s over the device), however deep the ring and however many
// workgroups share the CU, which is less than its matrix instructions could use at these tile sizes.  So the tile is as large
// as leaves one to a CU, and the ring as deep as LDS allows.  The barrier is a bare s_barrier behind a counted wait: __syncthreads()
// waits for every load into LDS first, and the ring degenerates to one step in flight (128 x 64 tiles, K = 5120: 67 us, now 39).
// LDS tile of an operand: row pairs form 256-byte lines, the 16-byte chunk c of row r sits in slot (r & 1) * 8 +
// (c ^ ((r >> 1) & 7)) of line r >> 1 — the 16 lanes of a b128 fragment read (16 consecutive rows, one chunk) then cover 256
// consecutive bytes' worth of banks, and a wave's load (1 KB: 8 rows) writes whole lines from whole 128-byte row pieces.
// K a multiple of 64; operands as f16 rows (16-byte aligned).
#define DL_STEP_ROW 128     // bytes of a row in one K step

template <int N>
__device__ __forceinline__ void wait_vmcnt() {                // s_waitcnt vmcnt(N) only (gfx9 encoding: expcnt and lgkmcnt at their maxima)
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

template <int N>
__device__ __forceinline__ void wait_vmcnt_lds() {            // s_waitcnt vmcnt(N) lgkmcnt(0)
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

template <int WN, int WM, int TI, int TJ, int NBUF, bool EMIT>
__device__ __forceinline__ void gemm_f16_tile_dl(const mm_args & a, int tiles_m, int tiles_n, int sw, int tile, const char * wb, const char * xb, char * db,
                                                 const epi_args & epi, int64_t batch_off, int64_t d_nb1) {
    constexpr int NW = WN * WM, BN = 32 * TI * WN, BM = 32 * TJ * WM;
    constexpr int XL = BN / (8 * NW), WL = BM / (8 * NW); static_assert(BN % (8 * NW) == 0 && BM % (8 * NW) == 0, "");          // 1 KB loads per wavefront and step (8 rows each)
    constexpr int STEP_BYTES = (BN + BM) * DL_STEP_ROW;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int per_col = sw * tiles_n, col = tile / per_col, rem = tile - col * per_col;
    const int cw = min(sw, tiles_m - col * sw);
    const int64_t m0 = (int64_t)(col * sw + rem % cw) * BM;
    const int64_t n0 = (int64_t)(rem / cw) * BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // load i of this wavefront covers rows 8 (NW i + wave) .. + 7 of the tile; this lane: row lrow of the 8, chunk lchunk
    const int lrow = 2 * (lane >> 4) + ((lane & 15) >> 3);
    const int lchunk = (lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7);
    const char * xp[XL]; const char * wp[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) { const int64_t n = n0 + 8 * (NW * i + wave) + lrow; xp[i] = xb + (n < a.N ? n : a.N - 1) * a.x_nb1 + lchunk * 16; }
#pragma unroll
    for (int i = 0; i < WL; ++i) { const int64_t m = m0 + 8 * (NW * i + wave) + lrow; wp[i] = wb + (m < a.M ? m : a.M - 1) * a.w_nb1 + lchunk * 16; }
    auto load = [&](int step, int buf) __attribute__((always_inline)) {
        const int64_t ko = (int64_t) step * DL_STEP_ROW;
        char * xs = smem + buf * STEP_BYTES + wave * 1024, * ws = xs + BN * DL_STEP_ROW;
#pragma unroll
        for (int i = 0; i < XL; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(xp[i] + ko), (__attribute__((address_space(3))) void *)(xs + i * (NW * 1024)), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < WL; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(wp[i] + ko), (__attribute__((address_space(3))) void *)(ws + i * (NW * 1024)), 16, 0, 0);
    };
    // The last NBUF - 1 steps have no later step to fetch: their loads bring the part of the GELU table that the epilogue wants,
    // or, without a GELU, one line again and again, so that the number of loads in flight stays what the waits count on.
    // Step KT - 1 lies in the last buffer, so the table grows from the first one on.
    const bool gelu = epi.flags & MI355X_EPI_GELU;
    auto load_table = [&](int s) __attribute__((always_inline)) {                // s-th of these steps
        constexpr int HALF = GELU_LDS_BYTES / 2048;      // 1 KB pieces of a half
        char * to = smem + s * STEP_BYTES + wave * 1024;
#pragma unroll
        for (int i = 0; i < XL + WL; ++i) {
            const int p = (s * (XL + WL) + i) * NW + wave;
            const char * t = (const char *) epi.gelu + (p < HALF ? p * 1024 : 0x8000 * 2 + (min(p, 2 * HALF - 1) - HALF) * 1024) + lane * 16;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(gelu ? t : wb), (__attribute__((address_space(3))) void *)(to + i * (NW * 1024)), 16, 0, 0);
        }
    };

    const int wn = (wave / WM) * 32 * TI, wmo = (wave % WM) * 32 * TJ;   // wave patch origin inside the tile
    const int l32 = lane & 31, g = lane >> 5;
    // fragment reads: row wn + 32 i + l32 (its line and half of the line), chunk 2 kk + g swizzled by the row
    const int rsw = (l32 >> 1) & 7;
    const int xrow = ((wn + l32) >> 1) * 256 + (l32 & 1) * 128, wrow = BN * DL_STEP_ROW + ((wmo + l32) >> 1) * 256 + (l32 & 1) * 128;
    int koff[GB_K / 16];
#pragma unroll
    for (int kk = 0; kk < GB_K / 16; ++kk) koff[kk] = ((2 * kk + g) ^ rsw) * 16;

    float16_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // One K step: all fragment reads of the step go out first (they return in order, so the matrix instructions start when
    // the first sub-step's have arrived and never wait for a read issued behind them); then the loads of a later step, one
    // behind each of the first matrix instructions — a load can sit in the issue stage while the CU's vector-memory path is
    // backed up, and everything behind it waits with it: spread out, a matrix instruction is already running each time
    // (1480 clocks per step instead of 1730 with the eight loads in front); then the rest of the 4 TI TJ matrix instructions.
    auto mma = [&](int buf, auto && fetch) __attribute__((always_inline)) {
        const char * xs = smem + buf * STEP_BYTES + xrow, * ws = smem + buf * STEP_BYTES + wrow;
        half8_t av[GB_K / 16][TI], bv[GB_K / 16][TJ];
#pragma unroll
        for (int kk = 0; kk < GB_K / 16; ++kk) {
#pragma unroll
            for (int i = 0; i < TI; ++i) av[kk][i] = *(const half8_t *)(xs + i * 4096 + koff[kk]);
#pragma unroll
            for (int j = 0; j < TJ; ++j) bv[kk][j] = *(const half8_t *)(ws + j * 4096 + koff[kk]);
        }
        fetch();
#pragma unroll
        for (int kk = 0; kk < GB_K / 16; ++kk)
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    // (EMIT: the patch transposed — rows are m, columns n — for the epilogue that writes the Q8_0-rounded image)
                    acc[i][j] = EMIT ? __builtin_amdgcn_mfma_f32_32x32x16_f16(bv[kk][j], av[kk][i], acc[i][j], 0, 0, 0)
                                     : __builtin_amdgcn_mfma_f32_32x32x16_f16(av[kk][i], bv[kk][j], acc[i][j], 0, 0, 0);
        constexpr int n_mma = (GB_K / 16) * TI * TJ, n_ld = XL + WL;
        static_assert(n_mma >= n_ld, "a matrix instruction in front of every load");
        __builtin_amdgcn_sched_group_barrier(0x100, (GB_K / 16) * (TI + TJ), 0);     // the DS reads
#pragma unroll
        for (int q = 0; q < n_ld; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                       // one matrix instruction,
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                       // one load
        }
        __builtin_amdgcn_sched_group_barrier(0x008, n_mma - n_ld, 0);                // the remaining matrix instructions
    };

    const int KT = (int)(a.K / GB_K), last = KT - 1;
    // Every step issues XL + WL loads, so "all but the (NBUF - 2) (XL + WL) youngest have landed" is a constant wait.
    int buf = (int)((uint32_t)(NBUF * KT - KT) % NBUF);         // of step 0: step KT - 1 lies in buffer NBUF - 1
    int fill = buf;
#pragma unroll
    for (int st = 0; st < NBUF - 1; ++st) { load(min(st, last), fill); fill = fill + 1 == NBUF ? 0 : fill + 1; }
    auto step_begins = [&]() __attribute__((always_inline)) {
        wait_vmcnt_lds<(NBUF - 2) * (XL + WL)>();         // this wavefront's pieces of the step are in LDS, its reads of the step before are done
        __builtin_amdgcn_s_barrier();                   // ... and everybody's.  (Not __syncthreads(), which waits for every load into LDS.)
        __builtin_amdgcn_sched_barrier(0);
    };
    const int kt_tail = max(KT - (NBUF - 1), 0);
    int kt = 0;
    for (; kt < kt_tail; ++kt) {
        step_begins();
        mma(buf, [&]() __attribute__((always_inline)) { load(kt + NBUF - 1, fill); });
        buf = buf + 1 == NBUF ? 0 : buf + 1; fill = fill + 1 == NBUF ? 0 : fill + 1;
    }
    const bool table = gelu && KT >= NBUF - 1;          // (a K shorter than the ring: the epilogue fetches the table)
    for (; kt < KT; ++kt) {
        step_begins();
        mma(buf, [&]() __attribute__((always_inline)) { load_table(kt - KT + NBUF - 1); });
        buf = buf + 1 == NBUF ? 0 : buf + 1;
    }
    wait_vmcnt<0>();
    __syncthreads();
    gemm_tile_epilogue<TI, TJ, EMIT, true, 64 * NW, BN, BM>(acc, a, epi, db, batch_off, d_nb1, n0, m0, wn, wmo, smem, table);
}

// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2: workgroup `lin` of `total` runs on XCD lin % 8.
// Give every XCD one run of consecutive work items, so that what its workgroups read is shared inside that L2: the index
// of this workgroup's item when XCD x takes items [x q + min(x, r), ...) with q = total / 8, r = total % 8.
__device__ __forceinline__ int xcd_run_index(int lin, int total) {
    const int xcd = lin % 8, q = total / 8, r = total % 8;
    return xcd * q + (xcd < r ? xcd : r) + lin / 8;
}

// width (in m-tiles) of the columns of the tile path: a run of `run` tiles should be as square as the tiles allow
static int tile_path_width(int64_t tiles_m, int64_t tiles_n, int64_t run, int bn, int bm) {
    if (run >= tiles_m * tiles_n || tiles_n == 1) return (int) tiles_m;
    int best = (int) tiles_m; int64_t best_cost = INT64_MAX;
    for (int64_t sw = 1; sw <= tiles_m; ++sw) {
        // rows of X and of W that a run touches (one more panel for a run that starts mid-way), more when the columns are uneven
        const int64_t cost = (std::min(tiles_n, (run + sw - 1) / sw + 1)) * bn + sw * bm + (tiles_m % sw ? bm : 0);
        if (cost < best_cost) { best_cost = cost; best = (int) sw; }
    }
    return best;
}

template <int TI, int TJ>
__global__ void __launch_bounds__(256, 2) k_gemm_f16(mm_args a, int tiles_m, int tiles_n, int sw) {
    const mm_slice_ptrs z = mm_slice(a, blockIdx.y);
    gemm_f16_tile<TI, TJ>(a, tiles_m, tiles_n, sw, xcd_run_index(blockIdx.x, tiles_m * tiles_n), z.w, z.x, a.d + z.d_off, a.e, z.d_off, a.d_nb1);
}

// LDS of the epilogue: the GELU table slice and, with an image, the rows on their way out
template <int NW, int TI, int TJ, bool EMIT> constexpr size_t dl_epilogue_bytes() { return GELU_LDS_BYTES + (EMIT ? (size_t) NW * 32 * TI * (64 * TJ + 16) : 0); }

template <int WN, int WM, int TI, int TJ, int NBUF, bool EMIT>
__global__ void __launch_bounds__(64 * WN * WM) k_gemm_f16_dl(mm_args a, int tiles_m, int tiles_n, int sw) {
    const mm_slice_ptrs z = mm_slice(a, blockIdx.y);
    gemm_f16_tile_dl<WN, WM, TI, TJ, NBUF, EMIT>(a, tiles_m, tiles_n, sw, xcd_run_index(blockIdx.x, tiles_m * tiles_n), z.w, z.x, a.d + z.d_off, a.e, z.d_off, a.d_nb1);
}
// Several products over the same src1 in one launch (the Q, K and V projections of a layer; the cross-attention K and V
// of all decoder layers): one launch of 3 x 80 or 64 x 60 tiles fills 256 CUs where 80 tiles at a time leave most of them idle.
// The products' tiles form one pool, product after product, and an XCD's run may cross from one product into the next.
template <int WN, int WM, int TI, int TJ, int NBUF>
__global__ void __launch_bounds__(64 * WN * WM) k_gemm_f16_dl_group(mm_args a, int tiles_m, int tiles_n, int sw, int count, mm_group grp) {
    const int nblk = tiles_m * tiles_n;
    const int item = xcd_run_index((int) blockIdx.x, nblk * count);
    const mm_group_entry & ge = grp.e[item / nblk];
    epi_args e;
    e.flags = ge.flags; e.scale = ge.scale; e.bias = ge.bias; e.residual = ge.residual; e.gelu = a.e.gelu; e.image = nullptr;
    gemm_f16_tile_dl<WN, WM, TI, TJ, NBUF, false>(a, tiles_m, tiles_n, sw, item % nblk, ge.w, a.x, ge.d, e, 0, ge.d_nb1);
}

// more than the default 64 KB of LDS have to be asked for, once per kernel and device
static int configure_lds(const void * fn, size_t lds, std::atomic<bool> * configured) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return MI355X_ERR_HIP;
    if (configured[dev].load(std::memory_order_acquire)) return MI355X_OK;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds) != hipSuccess) return MI355X_ERR_HIP;
    configured[dev].store(true, std::memory_order_release);
    return MI355X_OK;
}
struct tile_plan { int64_t tm, tn; int sw; dim3 grid; };
static int plan_tiles(const mm_args & a, int bn, int bm, int count, tile_plan & p) {
    p.tm = (a.M + bm - 1) / bm; p.tn = (a.N + bn - 1) / bn;
    if (p.tm * p.tn * count > 0x7fffffff || a.ne12 * a.ne13 > 65535) return MI355X_ERR_UNSUPPORTED;
    p.grid = dim3((unsigned)(p.tm * p.tn * count), (unsigned)(a.ne12 * a.ne13));
    p.sw = tile_path_width(p.tm, p.tn, (p.tm * p.tn * count + 7) / 8, bn, bm);
    return MI355X_OK;
}

// grp: the products of a group (count of them), NULL for one product
template <int WN, int WM, int TI, int TJ, int NBUF, bool EMIT>
static int launch_dl(const mm_args & a, const mm_group * grp, int count, hipStream_t st) {
    constexpr int BN = 32 * TI * WN, BM = 32 * TJ * WM;
    constexpr size_t lds = std::max((size_t) NBUF * (BN + BM) * DL_STEP_ROW, dl_epilogue_bytes<WN * WM, TI, TJ, EMIT>());
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    static std::atomic<bool> configured[64], group_configured[64];
    tile_plan p;
    if (int rc = plan_tiles(a, BN, BM, grp ? count : 1, p)) return rc;
    if constexpr (!EMIT) {
        if (grp) {
            if (int rc = configure_lds((const void *) k_gemm_f16_dl_group<WN, WM, TI, TJ, NBUF>, lds, group_configured)) return rc;
            k_gemm_f16_dl_group<WN, WM, TI, TJ, NBUF><<<p.grid, 64 * WN * WM, lds, st>>>(a, (int) p.tm, (int) p.tn, p.sw, count, *grp);
            return launch_status();
        }
    }
    if (int rc = configure_lds((const void *) k_gemm_f16_dl<WN, WM, TI, TJ, NBUF, EMIT>, lds, configured)) return rc;
    k_gemm_f16_dl<WN, WM, TI, TJ, NBUF, EMIT><<<p.grid, 64 * WN * WM, lds, st>>>(a, (int) p.tm, (int) p.tn, p.sw);
    return launch_status();
}
// The tile (n x m) by size: rounds of 256 tiles, one to a CU, times the rows of X and of W that a step of one fetches — 128 x 256 where
// they are one round (M = 5120, N = 1500: 33 us at K = 1280; 192 x 128 46, 128 x 128 39), 192 x 128 (M = 3840: 26; 28; 37 and M = 4096,
// 3072), 128 x 128 (M = 2048, K = 512: 10.7; 12.6 with 192 x 128, 13.5 with 128 x 64), 128 x 64 (M = 1280: 12.5; 16; 20).
enum { DL_128x256, DL_192x128, DL_128x128, DL_128x64 };
static int dl_pick(const mm_args & a, int count) {
    static const int bn[4] = { 128, 192, 128, 128 }, bm[4] = { 256, 128, 128, 64 };
    int best = DL_128x256; int64_t best_cost = INT64_MAX;
    for (int i = 0; i < 4; ++i) {
        const int64_t tiles = (a.N + bn[i] - 1) / bn[i] * ((a.M + bm[i] - 1) / bm[i]) * a.ne12 * a.ne13 * count, cost = (tiles + 255) / 256 * (bn[i] + bm[i]);
        if (cost < best_cost) { best_cost = cost; best = i; }
    }
    return best;
}
template <bool EMIT>
static int launch_gemm_f16_dl(const mm_args & a, const mm_group * grp, int count, hipStream_t st) {
    switch (dl_pick(a, count)) {
        case DL_128x256: return launch_dl<2, 4, 2, 2, 3, EMIT>(a, grp, count, st);
        case DL_192x128: return launch_dl<2, 4, 3, 1, 3, EMIT>(a, grp, count, st);
        case DL_128x128: return launch_dl<4, 2, 1, 2, 4, EMIT>(a, grp, count, st);
        default:         return launch_dl<4, 2, 1, 1, 6, EMIT>(a, grp, count, st);
    }
}

// the two-role form (K a multiple of 256)
#define RS_NP 512       // operand threads: 512 (three 16-byte pieces each per step of a 128 x 64 tile) beat 256 by 7 %
__global__ void __launch_bounds__(256 + RS_NP) k_gemm_f16_rs(mm_args a, int tiles_m, int tiles_n, int sw) {
    const mm_slice_ptrs z = mm_slice(a, blockIdx.y);
    gemm_f16_tile_rs<2, 1, 4, RS_NP>(a, tiles_m, tiles_n, sw, xcd_run_index(blockIdx.x, tiles_m * tiles_n), z.w, z.x, a.d + z.d_off, a.e, z.d_off, a.d_nb1);
}
static int launch_gemm_f16_rs(const mm_args & a, hipStream_t st) {
    constexpr size_t lds = (size_t) 2 * (128 + 64) * GB_LD * sizeof(half_t);
    tile_plan p;
    if (int rc = plan_tiles(a, 128, 64, 1, p)) return rc;
    k_gemm_f16_rs<<<p.grid, 256 + RS_NP, lds, st>>>(a, (int) p.tm, (int) p.tn, p.sw);
    return launch_status();
}

template <int TI, int TJ>
static int launch_gemm_f16(const mm_args & a, hipStream_t st) {
    constexpr int BN = 64 * TI, BM = 64 * TJ;
    constexpr size_t lds = (size_t) 2 * (BN + BM) * GB_LD * sizeof(half_t);
    static std::atomic<bool> configured[64];
    tile_plan p;
    if (int rc = plan_tiles(a, BN, BM, 1, p)) return rc;
    if (int rc = configure_lds((const void *) k_gemm_f16<TI, TJ>, lds, configured)) return rc;
    k_gemm_f16<TI, TJ><<<p.grid, 256, lds, st>>>(a, (int) p.tm, (int) p.tn, p.sw);
    return launch_status();
}

// Small problems go to k_gemm_ks; else K decides: a multiple of 64 goes over the direct loads.
static int launch_gemm_f16_auto(const mm_args & a, hipStream_t st) {
    const int64_t nb = a.ne12 * a.ne13;
    const bool emit = a.e.flags & MI355X_EPI_EMIT_F16;
    ks_shape ks;
    // (an image out of 64 x 64 tiles whose K is short: the 128-wide tiles have the better epilogue.  N = 700, M = 1280, K = 1280: 12.0 to
    // 13.2 us; N = 400, M = 3072, K = 768: 9.4; 13.5 — but K = 5120: 34; 28)
    if (ks_pick(a.M, a.N, a.K, nb, emit, ks) && !(emit && ks.mt == 4 && a.K < 2048)) return launch_gemm_ks(a, ks, KS_X_F16, nullptr, 0, st);
    static const bool staged = getenv("MI355X_GEMM_STAGED") != nullptr;        // the register-staged loop, for comparison
    if (a.K % GB_K == 0 && (!staged || emit)) {
        // a long K on 128 x 64 tiles, nothing but sums behind it: the two-role kernel (K = 3072, M = 768: 19 us, 21 over the direct loads)
        if (!emit && !(a.e.flags & MI355X_EPI_GELU) && a.K >= 2048 && a.K % (4 * GB_K) == 0 && dl_pick(a, 1) == DL_128x64) return launch_gemm_f16_rs(a, st);
        return emit ? launch_gemm_f16_dl<true>(a, nullptr, 1, st) : launch_gemm_f16_dl<false>(a, nullptr, 1, st);
    }
    if (emit) return MI355X_ERR_UNSUPPORTED;
    auto blocks = [&](int bn, int bm) { return ((a.N + bn - 1) / bn) * ((a.M + bm - 1) / bm) * nb; };
    if (blocks(128, 128) >= 384) return launch_gemm_f16<2, 2>(a, st);
    if (blocks(128, 64)  >= 192 || a.N > 64) return launch_gemm_f16<2, 1>(a, st);
    return launch_gemm_f16<1, 1>(a, st);       // (few tiles of a K that k_gemm_ks does not take)
}

// ------------------------------------------------------------------------------------------------------
// generic fallback: one wavefront per (m, group of up to 8 columns, batch); element-wise dequant, f32 FMA
// ------------------------------------------------------------------------------------------------------

__device__ __forceinline__ float w_elem(int type, const uint8_t * row, int64_t k) {
    switch (type) {
        case MI355X_TYPE_Q5_0: {
            const uint8_t * b = row + (k / QK) * 22; const int jj = (int)(k % QK);
            const float d = h2f(*(const uint16_t *) b);
            const uint32_t qh = *(const u32a2 *)(b + 2);
            const uint32_t qs = b[6 + (jj & 15)];
            const int nib = jj < 16 ? (qs & 0xF) : (qs >> 4);
            return (float)((nib | (((qh >> jj) & 1) << 4)) - 16) * d;
        }
        case MI355X_TYPE_Q8_0: {
            const uint8_t * b = row + (k / QK) * 34;
            return (float)((const int8_t *) b)[2 + k % QK] * h2f(*(const uint16_t *) b);
        }
        default:              return ((const float *) row)[k];
    }
}

__global__ void k_mul_mat_generic(mm_args a, int t0, int t1) {
    const int lane = threadIdx.x;
    const int64_t m  = blockIdx.x;
    const int64_t nb = (int64_t) blockIdx.y * 8;
    const int64_t b2 = blockIdx.z % a.ne12, b3 = blockIdx.z / a.ne12;
    const uint8_t * wrow = (const uint8_t *) a.w + m * a.w_nb1 + (b2 / a.r2) * a.w_nb2 + (b3 / a.r3) * a.w_nb3;
    const char * xb = a.x + b2 * a.x_nb2 + b3 * a.x_nb3;
    char * db = a.d + b2 * a.d_nb2 + b3 * a.d_nb3;
    float acc[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] = 0.0f;
    for (int64_t k = lane; k < a.K; k += WAVE) {
        const float w = w_elem(t0, wrow, k);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int64_t n = nb + c;
            if (n < a.N) {
                const char * xr = xb + n * a.x_nb1;
                const float x = t1 == MI355X_TYPE_F32 ? ((const float *) xr)[k] : (float)((const half_t *) xr)[k];
                acc[c] += w * x;
            }
        }
    }
    const bool out_f16 = a.e.flags & MI355X_EPI_OUT_F16;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float s = wave_sum(acc[c]);
        const int64_t n = nb + c;
        if (lane == 0 && n < a.N) {
            const float v = apply_epilogue(s, a.e, m, n, (b2 * a.d_nb2 + b3 * a.d_nb3) + n * a.d_nb1 + m * 4);
            if (out_f16) *(half_t *)(db + n * a.d_nb1 + m * 2) = (half_t) v;
            else         *(float  *)(db + n * a.d_nb1 + m * 4) = v;
        }
    }
}

// ------------------------------------------------------------------------------------------------------
// host dispatch
// ------------------------------------------------------------------------------------------------------



// which kernel a (src0, src1) pair runs on; depends on types, column count and alignment only
int mm_path(const mi355x_tensor * src0, const mi355x_tensor * src1) {
    const int t0 = src0->type, t1 = src1->type;
    const int64_t K = src0->ne[0], N = src1->ne[1];
    const int64_t nbatch = src1->ne[2] * src1->ne[3];
    const bool quant = blck_size(t0) > 1;
    const bool w_al2 = (uintptr_t) src0->data % 2 == 0 && src0->nb[1] % 2 == 0 && src0->nb[2] % 2 == 0 && src0->nb[3] % 2 == 0;

    // GEMV: few columns, quantized weights, plain 2-d problem, activations fit the LDS staging area
    if (quant && N <= MI355X_GEMV_MAX_COLS && nbatch == 1 && t1 == MI355X_TYPE_F32 && aligned16(src1) && w_al2 &&
        (size_t) N * K + (size_t) N * (K / QK) * 8 <= 64 * 1024) {
        return MM_GEMV;
    }
    bool fast = N > MI355X_GEMV_MAX_COLS || !quant;
    if (N <= 2) fast = false;                         // (one or two columns keep src1 at its precision)
    fast = fast && aligned16(src1) && K % 8 == 0;
    if (quant)                 fast = fast && w_al2;
    else if (t0 == MI355X_TYPE_F16) fast = fast && aligned16(src0);
    else                       fast = fast && aligned16(src0) && K % QK == 0;
    return fast ? MM_GEMM : MM_GENERIC;
}

extern "C" const char * mi355x_mul_mat_kernel_name(const mi355x_tensor * src0, const mi355x_tensor * src1) {
    if (!src0 || !src1) return "mul_mat.invalid";
    const int path = mm_path(src0, src1);
    switch (src0->type) {
        case MI355X_TYPE_Q5_0: return path == MM_GEMV ? "mul_mat.gemv_q5_0" : path == MM_GEMM ? "mul_mat.gemm_q5_0" : "mul_mat.generic_q5_0";
        case MI355X_TYPE_Q8_0: return path == MM_GEMV ? "mul_mat.gemv_q8_0" : path == MM_GEMM ? "mul_mat.gemm_q8_0" : "mul_mat.generic_q8_0";
        case MI355X_TYPE_F16:  return path == MM_GEMM ? "mul_mat.gemm_f16" : "mul_mat.generic_f16";
        default:               return path == MM_GEMM ? "mul_mat.gemm_f32" : "mul_mat.generic_f32";
    }
}

// workspace of the GEMM path: f16 image of src1 (when src1 is F32), then f16 image of src0 (when src0 is not F16), each
// batch slice rounded up to 256 bytes
static size_t x16_bytes(const mi355x_tensor * src1) {
    return src1->type == MI355X_TYPE_F32 ? round256((size_t) src1->ne[0] * src1->ne[1] * 2) * (size_t)(src1->ne[2] * src1->ne[3]) : 0;
}
static size_t w16_bytes(const mi355x_tensor * src0) {
    return src0->type != MI355X_TYPE_F16 ? round256((size_t) src0->ne[0] * src0->ne[1] * 2) * (size_t)(src0->ne[2] * src0->ne[3]) : 0;
}
extern "C" size_t mi355x_mul_mat_workspace_size(const mi355x_tensor * src0, const mi355x_tensor * src1) {
    if (!src0 || !src1) return 0;
    const int path = mm_path(src0, src1);
    if (path == MM_GEMV) return gemv_ws_bytes(src0, src1);
    if (path != MM_GEMM) return 0;
    return x16_bytes(src1) + w16_bytes(src0);
}

extern "C" int mi355x_mul_mat_group(const mi355x_mul_mat_item * items, int count, const mi355x_tensor * src1, int flags,
                                    void * workspace, size_t workspace_size, void * stream) {
    if (!items || !src1 || count < 1) return MI355X_ERR_INVALID;
    if (count > MM_GROUP_MAX) return MI355X_ERR_UNSUPPORTED;
    const mi355x_tensor * w0 = items[0].src0;
    if (!w0 || !items[0].dst) return MI355X_ERR_INVALID;
    if (blck_size(w0->type) > 1) return mul_mat_group_gemv(items, count, src1, flags, workspace, workspace_size, stream);
    // one shape of problem only: dense f16 weights (or weight images), 2-d, K a multiple of 256, the MFMA GEMM path
    if (w0->type != MI355X_TYPE_F16 || (src1->type != MI355X_TYPE_F32 && src1->type != MI355X_TYPE_F16)) return MI355X_ERR_UNSUPPORTED;
    if (src1->ne[2] != 1 || src1->ne[3] != 1 || w0->ne[2] != 1 || w0->ne[3] != 1) return MI355X_ERR_UNSUPPORTED;
    if (mm_path(w0, src1) != MM_GEMM || w0->ne[0] % (4 * GB_K) != 0) return MI355X_ERR_UNSUPPORTED;
    mm_args a;
    a.K = w0->ne[0]; a.M = w0->ne[1]; a.N = src1->ne[1];
    if (src1->ne[0] != a.K || w0->nb[0] != 2 || src1->nb[0] != type_size(src1->type)) return MI355X_ERR_INVALID;
    if (a.M == 0 || a.N == 0) return MI355X_OK;
    mm_group grp;
    bool any_gelu = false;
    for (int i = 0; i < count; ++i) {
        const mi355x_tensor * w = items[i].src0, * d = items[i].dst;
        const mi355x_epilogue * e = items[i].epi;
        if (!w || !d) return MI355X_ERR_INVALID;
        if (w->type != MI355X_TYPE_F16 || w->ne[0] != a.K || w->ne[1] != a.M || w->ne[2] != 1 || w->ne[3] != 1 || w->nb[0] != 2 || w->nb[1] != w0->nb[1] || !aligned16(w)) return MI355X_ERR_UNSUPPORTED;
        if (e && (e->flags & MI355X_EPI_EMIT_F16)) return MI355X_ERR_UNSUPPORTED;
        const int ef = e ? (e->flags & 63) : 0;
        const int td = (ef & MI355X_EPI_OUT_F16) ? MI355X_TYPE_F16 : MI355X_TYPE_F32;
        if (d->type != td || d->ne[0] != a.M || d->ne[1] != a.N || d->ne[2] != 1 || d->ne[3] != 1 || d->nb[0] != type_size(td) || d->nb[1] % 4 != 0) return MI355X_ERR_UNSUPPORTED;
        if ((ef & (MI355X_EPI_BIAS | MI355X_EPI_BIAS_COL)) && !e->bias) return MI355X_ERR_INVALID;
        if ((ef & MI355X_EPI_BIAS) && (ef & MI355X_EPI_BIAS_COL)) return MI355X_ERR_INVALID;
        if ((ef & MI355X_EPI_RESIDUAL) && (!e->residual || (ef & MI355X_EPI_OUT_F16))) return MI355X_ERR_INVALID;
        any_gelu = any_gelu || (ef & MI355X_EPI_GELU);
        grp.e[i] = { (const char *) w->data, (char *) d->data, e ? (const float *) e->bias : nullptr, e ? (const char *) e->residual : nullptr, (int64_t) d->nb[1], ef, e ? e->scale : 1.0f };
    }
    a.w = (const char *) w0->data; a.x = (const char *) src1->data; a.d = (char *) items[0].dst->data;
    a.w_nb1 = w0->nb[1]; a.w_nb2 = a.w_nb3 = 0;
    a.x_nb1 = src1->nb[1]; a.x_nb2 = a.x_nb3 = 0;
    a.d_nb1 = items[0].dst->nb[1]; a.d_nb2 = a.d_nb3 = 0;
    a.ne12 = a.ne13 = a.r2 = a.r3 = 1;
    a.e.flags = 0; a.e.scale = 1.0f; a.e.bias = nullptr; a.e.residual = nullptr; a.e.gelu = nullptr; a.e.image = nullptr;
    if (any_gelu && !(a.e.gelu = gelu_table_device())) return MI355X_ERR_HIP;
    hipStream_t st = (hipStream_t) stream;

    const size_t xbytes = x16_bytes(src1);
    if (xbytes) {
        if (!workspace || workspace_size < xbytes || (uintptr_t) workspace % 256 != 0) return MI355X_ERR_WORKSPACE;
        if (!(flags & MI355X_MM_WS_READY)) {
            dim3 qgrid((unsigned)((a.K / 4 * a.N + 255) / 256), 1);
            const bool q8 = (flags & MI355X_MM_ACT_Q8_0) && !(flags & MI355X_MM_EXACT_ACT);
            // a handful of columns: the products round src1 to f16 themselves, the first leaves the rows in the workspace
            ks_shape ks;
            if (!q8 && !(flags & MI355X_MM_PREPARE_ONLY) && ks_pick_group(a.M, a.N, a.K, count, ks) && ks_converts(ks))
                return launch_gemm_ks_group(a, grp, count, ks, (half_t *) workspace, st);
            if (q8) k_x_to_f16<true ><<<qgrid, 256, 0, st>>>(a.x, (half_t *) workspace, a.K, a.N, a.x_nb1, 0, 1, 0, 0);
            else    k_x_to_f16<false><<<qgrid, 256, 0, st>>>(a.x, (half_t *) workspace, a.K, a.N, a.x_nb1, 0, 1, 0, 0);
        }
        a.x = (const char *) workspace; a.x_nb1 = a.K * 2;
    }
    if (flags & MI355X_MM_PREPARE_ONLY) return launch_status();
    ks_shape ks;
    if (ks_pick_group(a.M, a.N, a.K, count, ks)) return launch_gemm_ks_group(a, grp, count, ks, nullptr, st);
    return launch_gemm_f16_dl<false>(a, &grp, count, st);
}

extern "C" int mi355x_dequantize_row_f16(int type, const void * src, void * dst, int64_t k, void * stream) {
    if (!src || !dst || k < 0 || k % QK != 0 || (uintptr_t) src % 2 != 0 || (uintptr_t) dst % 16 != 0) return MI355X_ERR_INVALID;
    if (k == 0) return MI355X_OK;
    if (k / QK > 0x7fffffff * (int64_t) 256) return MI355X_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t) stream;
    const unsigned grid = (unsigned)((k / QK + 255) / 256);
    if      (type == MI355X_TYPE_Q5_0) k_w_to_f16<MI355X_TYPE_Q5_0><<<grid, 256, 0, st>>>((const char *) src, (half_t *) dst, k, 1, 0, 0, 1, 0, 0);
    else if (type == MI355X_TYPE_Q8_0) k_w_to_f16<MI355X_TYPE_Q8_0><<<grid, 256, 0, st>>>((const char *) src, (half_t *) dst, k, 1, 0, 0, 1, 0, 0);
    else return MI355X_ERR_UNSUPPORTED;
    return launch_status();
}

extern "C" int mi355x_mul_mat(const mi355x_tensor * src0, const mi355x_tensor * src1, const mi355x_tensor * dst,
                              const mi355x_epilogue * epi, void * workspace, size_t workspace_size, void * stream) {
    if (!src0 || !src1 || !dst) return MI355X_ERR_INVALID;
    const int t0 = src0->type, t1 = src1->type;
    if (t0 != MI355X_TYPE_Q5_0 && t0 != MI355X_TYPE_Q8_0 && t0 != MI355X_TYPE_F16 && t0 != MI355X_TYPE_F32) return MI355X_ERR_UNSUPPORTED;
    if (t1 != MI355X_TYPE_F32 && t1 != MI355X_TYPE_F16) return MI355X_ERR_UNSUPPORTED;
    const int flags = epi ? epi->flags : 0;
    const int td = (flags & MI355X_EPI_OUT_F16) ? MI355X_TYPE_F16 : MI355X_TYPE_F32;
    if (dst->type != td) return MI355X_ERR_INVALID;

    mm_args a;
    a.K = src0->ne[0]; a.M = src0->ne[1]; a.N = src1->ne[1];
    if (src1->ne[0] != a.K || dst->ne[0] != a.M || dst->ne[1] != a.N) return MI355X_ERR_INVALID;
    if (dst->ne[2] != src1->ne[2] || dst->ne[3] != src1->ne[3]) return MI355X_ERR_INVALID;
    if (src0->ne[2] <= 0 || src0->ne[3] <= 0 || src1->ne[2] % src0->ne[2] != 0 || src1->ne[3] % src0->ne[3] != 0) return MI355X_ERR_INVALID;
    if (src0->nb[0] != type_size(t0) || src1->nb[0] != type_size(t1) || dst->nb[0] != type_size(td)) return MI355X_ERR_UNSUPPORTED;
    if (blck_size(t0) > 1 && a.K % QK != 0) return MI355X_ERR_INVALID;
    if ((flags & (MI355X_EPI_BIAS | MI355X_EPI_BIAS_COL)) && !epi->bias) return MI355X_ERR_INVALID;
    if ((flags & MI355X_EPI_BIAS) && (flags & MI355X_EPI_BIAS_COL)) return MI355X_ERR_INVALID;      // there is one bias pointer
    if ((flags & MI355X_EPI_RESIDUAL) && !epi->residual) return MI355X_ERR_INVALID;
    if ((flags & MI355X_EPI_RESIDUAL) && (flags & MI355X_EPI_OUT_F16)) return MI355X_ERR_UNSUPPORTED;
    if (a.M == 0 || a.N == 0 || dst->ne[2] * dst->ne[3] == 0) return MI355X_OK;
    if ((flags & MI355X_MM_PREPARE_ONLY) && mm_path(src0, src1) == MM_GENERIC) return MI355X_OK;   // nothing to prepare

    a.w = (const char *) src0->data; a.x = (const char *) src1->data; a.d = (char *) dst->data;
    a.w_nb1 = src0->nb[1]; a.w_nb2 = src0->nb[2]; a.w_nb3 = src0->nb[3];
    a.x_nb1 = src1->nb[1]; a.x_nb2 = src1->nb[2]; a.x_nb3 = src1->nb[3];
    a.d_nb1 = dst->nb[1];  a.d_nb2 = dst->nb[2];  a.d_nb3 = dst->nb[3];
    a.ne12 = src1->ne[2]; a.ne13 = src1->ne[3];
    a.r2 = src1->ne[2] / src0->ne[2]; a.r3 = src1->ne[3] / src0->ne[3];
    a.e.flags = flags; a.e.scale = epi ? epi->scale : 1.0f;
    a.e.bias = epi ? (const float *) epi->bias : nullptr;
    a.e.residual = epi ? (const char *) epi->residual : nullptr;
    a.e.gelu = nullptr;
    if ((flags & MI355X_EPI_GELU) && !(a.e.gelu = gelu_table_device())) return MI355X_ERR_HIP;
    a.e.image = epi ? (half_t *) epi->image : nullptr;
    if (flags & MI355X_EPI_EMIT_F16) {
        if (!a.e.image || (flags & MI355X_EPI_OUT_F16)) return MI355X_ERR_INVALID;
    }
    if ((flags & MI355X_EPI_IMAGE_ONLY) && !(flags & MI355X_EPI_EMIT_F16)) return MI355X_ERR_INVALID;
    if (flags & MI355X_EPI_EMIT_Q8_0) {                       // the register kernel of the few-column path only
        if (!a.e.image || (uintptr_t) a.e.image % 16 != 0 || (flags & (MI355X_EPI_OUT_F16 | MI355X_EPI_EMIT_F16))) return MI355X_ERR_INVALID;
        const size_t ws_need = gemv_ws_bytes(src0, src1);
        if (a.M % QK != 0 || mm_path(src0, src1) != MM_GEMV || !ws_need || !workspace || workspace_size < ws_need || (uintptr_t) workspace % 16 != 0) return MI355X_ERR_UNSUPPORTED;
    }
    if (flags & MI355X_EPI_EMIT_F16) {
        if (a.M % QK != 0 || dst->ne[2] * dst->ne[3] != 1 || mm_path(src0, src1) != MM_GEMM) return MI355X_ERR_UNSUPPORTED;
    }

    hipStream_t st = (hipStream_t) stream;
    const int64_t nbatch = a.ne12 * a.ne13;
    if (nbatch > 65535) return MI355X_ERR_UNSUPPORTED;

    const int path = mm_path(src0, src1);
    const bool quant = blck_size(t0) > 1;
    if (path == MM_GEMV) {
        // with a workspace: activations quantized once (skipped when the caller says they are there), then the product
        // with them in registers; without: every workgroup quantizes them into LDS for itself
        const size_t need = gemv_ws_bytes(src0, src1);
        if (need && workspace && workspace_size >= need && (uintptr_t) workspace % 16 == 0) {
            if (!(flags & MI355X_MM_WS_READY)) {
                if (const int rc = launch_quantize_x_q8(a.x, a.x_nb1, a.K, a.N, (char *) workspace, st)) return rc;
            }
            if (flags & MI355X_MM_PREPARE_ONLY) return MI355X_OK;
            mm_args g = a;
            g.x = (const char *) workspace;
            return launch_gemv_ws(t0, g, st);
        }
        if (flags & MI355X_MM_PREPARE_ONLY) return MI355X_OK;
        return launch_gemv_lds(t0, a, st);
    }
    if (path == MM_GEMM) {
        const size_t xbytes = x16_bytes(src1), wbytes = w16_bytes(src0);
        if (xbytes + wbytes > 0 && (!workspace || workspace_size < xbytes + wbytes || (uintptr_t) workspace % 256 != 0)) return MI355X_ERR_WORKSPACE;
        mm_args g = a;
        if (xbytes) {
            const int64_t slice = (int64_t) round256((size_t)(a.N * a.K * 2));
            if (!(flags & MI355X_MM_WS_READY)) {
                dim3 qgrid((unsigned)((a.K / 4 * a.N + 255) / 256), (unsigned) nbatch);
                const bool q8 = (quant || (flags & MI355X_MM_ACT_Q8_0)) && !(flags & MI355X_MM_EXACT_ACT);
                if (q8 && a.K % QK != 0) return MI355X_ERR_INVALID;
                // a handful of columns: the product rounds src1 to f16 itself and leaves the f16 rows in the workspace on the way
                ks_shape ks;
                if (!q8 && !wbytes && !(flags & (MI355X_MM_PREPARE_ONLY | MI355X_EPI_EMIT_F16)) && ks_pick(a.M, a.N, a.K, nbatch, false, ks) && ks_converts(ks))
                    return launch_gemm_ks(a, ks, KS_X_CVT, (half_t *) workspace, slice / 2, st);
                if (q8) k_x_to_f16<true ><<<qgrid, 256, 0, st>>>(a.x, (half_t *) workspace, a.K, a.N, a.x_nb1, a.x_nb2, a.ne12, a.x_nb3, slice / 2);
                else    k_x_to_f16<false><<<qgrid, 256, 0, st>>>(a.x, (half_t *) workspace, a.K, a.N, a.x_nb1, a.x_nb2, a.ne12, a.x_nb3, slice / 2);
            }
            g.x = (const char *) workspace; g.x_nb1 = a.K * 2; g.x_nb2 = slice; g.x_nb3 = slice * a.ne12;
        }
        if (flags & MI355X_MM_PREPARE_ONLY) return launch_status();
        if (wbytes) {
            const int64_t slice = (int64_t) round256((size_t)(a.M * a.K * 2));
            half_t * w16 = (half_t *)((char *) workspace + xbytes);
            dim3 wgrid((unsigned)((a.K / QK * a.M + 255) / 256), (unsigned)(src0->ne[2] * src0->ne[3]));
            switch (t0) {
                case MI355X_TYPE_Q5_0: k_w_to_f16<MI355X_TYPE_Q5_0><<<wgrid, 256, 0, st>>>(a.w, w16, a.K, a.M, a.w_nb1, a.w_nb2, src0->ne[2], a.w_nb3, slice / 2); break;
                case MI355X_TYPE_Q8_0: k_w_to_f16<MI355X_TYPE_Q8_0><<<wgrid, 256, 0, st>>>(a.w, w16, a.K, a.M, a.w_nb1, a.w_nb2, src0->ne[2], a.w_nb3, slice / 2); break;
                default:               k_w_to_f16<MI355X_TYPE_F32 ><<<wgrid, 256, 0, st>>>(a.w, w16, a.K, a.M, a.w_nb1, a.w_nb2, src0->ne[2], a.w_nb3, slice / 2); break;
            }
            g.w = (const char *) w16; g.w_nb1 = a.K * 2; g.w_nb2 = slice; g.w_nb3 = slice * src0->ne[2];
        }
        return launch_gemm_f16_auto(g, st);
    }

    // f16 weights that the tiled kernels do not take: one or two columns, or rows that are not 16-byte aligned (the product of
    // the attention probabilities with the transposed V, whose rows have the length of the window).  src1 keeps its precision.
    if (t0 == MI355X_TYPE_F16) {
        ks_shape ks;
        if (t1 == MI355X_TYPE_F32 && a.N <= 2 && aligned16(src0) && aligned16(src1) && ks_pick(a.M, a.N, a.K, nbatch, false, ks)) return launch_gemm_ks(a, ks, KS_X_F32, nullptr, 0, st);
        return launch_gemm_kd(a, t1 == MI355X_TYPE_F32 ? KS_X_F32 : KS_X_F16, st);
    }
    if (a.M > 0x7fffffff || (a.N + 7) / 8 > 65535) return MI355X_ERR_UNSUPPORTED;
    dim3 grid((unsigned) a.M, (unsigned)((a.N + 7) / 8), (unsigned) nbatch);
    k_mul_mat_generic<<<grid, WAVE, 0, st>>>(a, t0, t1);
    return launch_status();
}

// ------------------------------------------------------------------------------------------------------
// mi355x_mul_mat for callers that cannot allocate (code under HIP graph capture, serving loops, harnesses that forbid
// hipMalloc): the workspace is a fixed array in device memory that belongs to the library, one copy per GPU.
// ------------------------------------------------------------------------------------------------------

#define MM_SCRATCH_BYTES (32u << 20)

static __device__ __align__(256) unsigned char scratch[MM_SCRATCH_BYTES];

// The array's device address on the current device (each GPU holds its own copy at its own address), looked up once per
// device with that device current.  `scratch` itself is only a host-side handle: host code never passes it to a kernel
// or a copy, always this pointer.
static void * scratch_on_current_device() {
    static std::mutex mu;
    static void * ptr[64] = {};
    static bool   failed[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) { (void) hipGetLastError(); return nullptr; }
    std::lock_guard<std::mutex> lock(mu);
    if (ptr[dev] || failed[dev]) return ptr[dev];
    void * p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) { (void) hipGetLastError(); failed[dev] = true; return nullptr; }
    ptr[dev] = p;
    return p;
}

extern "C" int mi355x_mul_mat_noalloc(const mi355x_tensor * src0, const mi355x_tensor * src1, const mi355x_tensor * dst,
                                      const mi355x_epilogue * epi, void * stream) {
    if (!src0 || !src1 || !dst) return MI355X_ERR_INVALID;
    // the array keeps whatever the call before left in it: nothing may claim that it already holds this call's activations
    if (epi && (epi->flags & (MI355X_MM_WS_READY | MI355X_MM_PREPARE_ONLY))) return MI355X_ERR_INVALID;
    const size_t need = mi355x_mul_mat_workspace_size(src0, src1);
    if (need > MM_SCRATCH_BYTES) return MI355X_ERR_WORKSPACE;         // beyond the array: use mi355x_mul_mat with a workspace of the caller's
    void * ws = scratch_on_current_device();
    if (!ws) return MI355X_ERR_HIP;
    // every byte a kernel of this call reads from the array is written by this call's own conversion pass first, so
    // nothing needs clearing
    return mi355x_mul_mat(src0, src1, dst, epi, ws, MM_SCRATCH_BYTES, stream);
}

