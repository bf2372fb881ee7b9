// MUL_MAT over Q5_0 / Q8_0 weights with at most 8 columns (a decode step): src1 is quantized to Q8_0 exactly as the CPU backend
// does before its dot products (quantize_row_q8_0, ggml-cpu-quants.c:808-865; ggml-cpu.c:1328-1363), and integer block dot
// products are scaled by d_w * d_x like ggml_vec_dot_q8_0_q8_0 / ggml_vec_dot_q5_0_q8_0 (ggml-cpu-quants.c:3597, 2930).
#include "gemv.h"
#include "gemv_q8_0_tiles.h"

#include <algorithm>
#include <type_traits>

// ------------------------------------------------------------------------------------------------------
// quantized GEMV (N <= 8)
// ------------------------------------------------------------------------------------------------------

// one weight block as loaded: scale bits, (Q5_0: high bits,) quants
template <int T0> struct wraw { uint32_t d, qh, q[T0 == MI355X_TYPE_Q8_0 ? 8 : 4]; };
template <int T0>
__device__ __forceinline__ wraw<T0> load_wraw(const uint8_t * wrow, int kb) {
    wraw<T0> r;
    if constexpr (T0 == MI355X_TYPE_Q8_0) {
        const uint8_t * b = wrow + (int64_t) kb * 34;
        r.d = *(const uint16_t *) b; r.qh = 0;
        const u128a2 q0 = *(const u128a2 *)(b + 2), q1 = *(const u128a2 *)(b + 18);
        r.q[0] = q0.x; r.q[1] = q0.y; r.q[2] = q0.z; r.q[3] = q0.w; r.q[4] = q1.x; r.q[5] = q1.y; r.q[6] = q1.z; r.q[7] = q1.w;
    } else {
        const uint8_t * b = wrow + (int64_t) kb * 22;
        r.d = *(const uint16_t *) b; r.qh = *(const u32a2 *)(b + 2);
        const u128a2 qs = *(const u128a2 *)(b + 6);
        r.q[0] = qs.x; r.q[1] = qs.y; r.q[2] = qs.z; r.q[3] = qs.w;
    }
    return r;
}

// X -> Q8_0 in LDS (int32 xq[NC][K/4] | float xd[NC][K/32] | int32 xsum[NC][K/32]) by the 256 threads of a workgroup
template <int NC>
__device__ __forceinline__ void quantize_x_to_lds(const mm_args & a, int32_t * xq, float * xd, int32_t * xsum, int nbk) {
    const int64_t K = a.K;
    // --- quantize X: 8 lanes per 32-value block, round-to-nearest-even like _mm256_round_ps(_MM_ROUND_NEAREST).
    // Eight independent loads per thread are in flight before the first is consumed.
    {
        const int total = NC * nbk * 8;                         // float4 pieces
        const int k8 = nbk * 8;
        for (int base = 0; base < total; base += 256 * 8) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int idx = base + u * 256 + (int) threadIdx.x;
                v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (idx < total) v[u] = *(const float4 *)(a.x + (int64_t)(idx / k8) * a.x_nb1 + (int64_t)(idx % k8) * 16);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int idx = base + u * 256 + (int) threadIdx.x;      // lanes 8i .. 8i+7 share a block
                float amax = fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
                amax = lanes_max<8>(amax);
                const float d  = div127(amax);
                const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
                const int q0 = (int) rintf(v[u].x * id), q1 = (int) rintf(v[u].y * id), q2 = (int) rintf(v[u].z * id), q3 = (int) rintf(v[u].w * id);
                int sum = q0 + q1 + q2 + q3;
                sum = lanes_sum<8>(sum);
                if (idx < total) {
                    const int n = idx / k8, c = idx % k8;       // c: float4 piece within the row
                    xq[(int64_t) n * (K / 4) + c] = (q0 & 0xFF) | ((q1 & 0xFF) << 8) | ((q2 & 0xFF) << 16) | ((q3 & 0xFF) << 24);
                    if ((c & 7) == 0) {
                        xd[n * nbk + c / 8]   = h2f(f2h_bits(d));     // the CPU backend stores d as f16 and reads it back
                        xsum[n * nbk + c / 8] = sum;
                    }
                }
            }
        }
    }
}

// LDS: int32 xq[NC][K/4] | float xd[NC][K/32] | int32 xsum[NC][K/32]
template <int T0, int NC, int LPR>
__global__ void __launch_bounds__(256) k_gemv_q(mm_args a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int64_t K = a.K;
    const int nbk = (int)(K / QK);
    int32_t * xq   = (int32_t *) smem;
    float *   xd   = (float *)(smem + (size_t) NC * K);
    int32_t * xsum = (int32_t *)(smem + (size_t) NC * K + (size_t) NC * nbk * 4);

    // A workgroup takes every gridDim.x-th group of 4 * (64 / LPR) rows; the activations are quantized once for all of them.
    constexpr int RPW = WAVE / LPR;                 // rows per wavefront
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane % LPR, r = lane / LPR;
    const int64_t n_groups = (a.M + 4 * RPW - 1) / (4 * RPW);
    int64_t group = blockIdx.x;
    int64_t row = group * (4 * RPW) + wave * RPW + r;
    bool row_ok = row < a.M;
    const uint8_t * wrow = (const uint8_t *) a.w + (row_ok ? row : 0) * a.w_nb1;

    // the epilogue operands of the lane that will store are fetched early, under the weight stream
    float e_bias = 0.0f, e_bcol[NC], e_res[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) { e_bcol[n] = 0.0f; e_res[n] = 0.0f; }
    auto fetch_epilogue = [&]() __attribute__((always_inline)) {
        if (row_ok && j == 0) {
            if (a.e.flags & MI355X_EPI_BIAS) e_bias = a.e.bias[row];
            if (a.e.flags & MI355X_EPI_BIAS_COL) {
#pragma unroll
                for (int n = 0; n < NC; ++n) e_bcol[n] = a.e.bias[n];
            }
            if (a.e.flags & MI355X_EPI_RESIDUAL) {
#pragma unroll
                for (int n = 0; n < NC; ++n) e_res[n] = *(const float *)(a.e.residual + n * a.d_nb1 + row * 4);
            }
        }
    };
    fetch_epilogue();

    // this lane's first weight block is requested before the activations are touched: the two HBM round trips of the
    // kernel (activations, weights) overlap instead of following each other
    wraw<T0> blk;
    if (row_ok && j < nbk) blk = load_wraw<T0>(wrow, j);

    quantize_x_to_lds<NC>(a, xq, xd, xsum, nbk);
    __syncthreads();

    for (;;) {
        float acc[NC];
#pragma unroll
        for (int n = 0; n < NC; ++n) acc[n] = 0.0f;
        if (row_ok) {
            for (int kb = j; kb < nbk; kb += LPR) {
                const wraw<T0> cur = blk;
                if (kb + LPR < nbk) blk = load_wraw<T0>(wrow, kb + LPR);      // next block in flight under this one's dot products
                uint32_t q[8];
                const float dw = h2f((uint16_t) cur.d);
                if constexpr (T0 == MI355X_TYPE_Q8_0) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) q[i] = cur.q[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {     // unsigned 5-bit values; the -16 is applied through xsum
                        q[i]     = (cur.q[i] & 0x0F0F0F0Fu)        | spread4_to_bit4((cur.qh >> (4*i))      & 0xFu);
                        q[4 + i] = ((cur.q[i] >> 4) & 0x0F0F0F0Fu) | spread4_to_bit4((cur.qh >> (16 + 4*i)) & 0xFu);
                    }
                }
#pragma unroll
                for (int n = 0; n < NC; ++n) {
                    const int4 x0 = *(const int4 *)(xq + (int64_t) n * (K / 4) + kb * 8);
                    const int4 x1 = *(const int4 *)(xq + (int64_t) n * (K / 4) + kb * 8 + 4);
                    int s = 0;
                    s = __builtin_amdgcn_sdot4((int) q[0], x0.x, s, false);
                    s = __builtin_amdgcn_sdot4((int) q[1], x0.y, s, false);
                    s = __builtin_amdgcn_sdot4((int) q[2], x0.z, s, false);
                    s = __builtin_amdgcn_sdot4((int) q[3], x0.w, s, false);
                    s = __builtin_amdgcn_sdot4((int) q[4], x1.x, s, false);
                    s = __builtin_amdgcn_sdot4((int) q[5], x1.y, s, false);
                    s = __builtin_amdgcn_sdot4((int) q[6], x1.z, s, false);
                    s = __builtin_amdgcn_sdot4((int) q[7], x1.w, s, false);
                    if constexpr (T0 == MI355X_TYPE_Q5_0) s -= 16 * xsum[n * nbk + kb];
                    acc[n] += (float) s * (dw * xd[n * nbk + kb]);
                }
            }
        }
        // this group's results are complete in registers; request the next group's first block before reducing and storing
        const int64_t done_row = row;
        const bool done_writer = row_ok && j == 0;
        const float o_bias = e_bias;
        float o_bcol[NC], o_res[NC];
#pragma unroll
        for (int n = 0; n < NC; ++n) { o_bcol[n] = e_bcol[n]; o_res[n] = e_res[n]; }
        group += gridDim.x;
        const bool more = group < n_groups;                 // uniform
        if (more) {
            row = group * (4 * RPW) + wave * RPW + r;
            row_ok = row < a.M;
            wrow = (const uint8_t *) a.w + (row_ok ? row : 0) * a.w_nb1;
            if (row_ok && j < nbk) blk = load_wraw<T0>(wrow, j);
            fetch_epilogue();
        }
#pragma unroll
        for (int n = 0; n < NC; ++n) {
#pragma unroll
            for (int o = LPR / 2; o > 0; o >>= 1) acc[n] += __shfl_xor(acc[n], o, LPR);
        }
        if (done_writer) {
            const bool out_f16 = a.e.flags & MI355X_EPI_OUT_F16;
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                float v = acc[n] + o_bias + o_bcol[n];          // at most one of the two biases is set
                if (a.e.flags & MI355X_EPI_GELU)     v  = gelu_f32(v, a.e.gelu);
                if (a.e.flags & MI355X_EPI_SCALE)    v *= a.e.scale;
                if (a.e.flags & MI355X_EPI_RESIDUAL) v += o_res[n];
                if (out_f16) *(half_t *)(a.d + n * a.d_nb1 + done_row * 2) = (half_t) v;
                else         *(float  *)(a.d + n * a.d_nb1 + done_row * 4) = v;
            }
        }
        if (!more) break;
    }
}

// Activations quantized ahead of the product, once for every product that reads them:
//   int8 xq[N][K] | float xd[N][K/32] (the f16-rounded block scales) | int32 xsum[N][K/32] (sum of a block's quants)
// One thread per four values, eight lanes per block; rounding as quantize_row_q8_0 (ggml-cpu-quants.c:808-865).
__global__ void __launch_bounds__(256) k_quantize_x_q8(const char * __restrict__ x, int64_t x_nb1, int64_t K, int64_t N, char * __restrict__ ws) {
    const int64_t k4 = K / 4, nbk = K / QK;
    const int64_t idx = (int64_t) blockIdx.x * 256 + threadIdx.x;          // K % 32 == 0: the 8 lanes of a block are in or out together
    if (idx >= N * k4) return;
    const int64_t n = idx / k4, c = idx % k4;
    const float4 v = *(const float4 *)(x + n * x_nb1 + c * 16);
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    amax = lanes_max<8>(amax);
    const float d  = div127(amax);
    const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
    const int q0 = (int) rintf(v.x * id), q1 = (int) rintf(v.y * id), q2 = (int) rintf(v.z * id), q3 = (int) rintf(v.w * id);
    int sum = q0 + q1 + q2 + q3;
    sum = lanes_sum<8>(sum);
    int32_t * xq   = (int32_t *) ws;
    float *   xd   = (float *)(ws + N * K);
    int32_t * xsum = (int32_t *)(ws + N * K + N * nbk * 4);
    xq[n * k4 + c] = (q0 & 0xFF) | ((q1 & 0xFF) << 8) | ((q2 & 0xFF) << 16) | ((q3 & 0xFF) << 24);
    if ((c & 7) == 0) {
        xd[n * nbk + c / 8]   = h2f(f2h_bits(d));          // the CPU backend stores d as f16 and reads it back
        xsum[n * nbk + c / 8] = sum;
    }
}

// rows of a launch up to which a product is a matter of latency (a layer's products; a vocabulary is a stream)
#define GEMV_SHORT_ROWS 16384
// lanes per row there: a block of 32 weights per lane (K <= 2048)
static constexpr int gemv_row_lanes(int nbk) { return nbk <= 16 ? 16 : nbk <= 32 ? 32 : 64; }

// The product over activations quantized ahead (a.x: the layout above, NC rows).  Lane j of a row's LPR lanes owns blocks
// j, j + LPR, ... (NB of them) of EVERY row it visits, so its slices of the activations are read once and stay in
// registers while the workgroup walks its row groups: the loop is weight loads and integer dot products only.  With
// the activations in LDS, their reads (NC x 32 bytes per 34-byte block) are what bounds the kernel, and quantizing them
// in every workgroup costs more than the product itself once K is large.
//
// `prologue`: what makes those activations, when they are not in the workspace yet (the fused LayerNorm leaves them in LDS).
// Its wavefronts request their rows BEFORE their first weight blocks (request(); request_late(), if there is one, the loads
// whose addresses those fetched, after the weight blocks) and finish() waits for the rows only: loads are waited for in the
// order they were issued, so the LayerNorm's reductions run while the weight blocks are on their way.  Wavefronts without a row
// go straight to their weights: the two sides of the branch request them separately, because a load behind a join is waited for
// as if it had been issued last.
struct gemv_no_prologue {
    static constexpr int ROWS = 0;                  // wavefronts that have a row to normalize
    static constexpr bool LATE = false;
    __device__ __forceinline__ void request() {}
    __device__ __forceinline__ void request_late() {}
    __device__ __forceinline__ void finish() {}
    __device__ __forceinline__ const char * publish(const char * x) { return x; }
};

//
// walk: how the workgroups share the row groups, worked out by the host (the size of the workgroup or of the grid is a trip to
// memory of its own on the device, and a division a hundred instructions)
struct gemv_walk {
    int waves_log2;      // wavefronts of a workgroup
    int n_groups;        // groups of rows, each what a workgroup's wavefronts do at a time
    int step;            // groups between two of a workgroup (the grid; 1 with the Q8_0 emission)
    int run;             // Q8_0 emission: groups of a workgroup, else 0
};

template <int T0, int NC, int LPR, int NB, int W_MAX, typename PRO = gemv_no_prologue>
__device__ __forceinline__ void gemv_qr_rows(const mm_args & a, const gemv_walk & walk, PRO prologue = PRO()) {
    const int64_t K = a.K;
    const int nbk = (int)(K / QK);

    constexpr int RPW = WAVE / LPR;                 // rows per wavefront
    constexpr int RPW_LOG2 = LPR == 16 ? 2 : LPR == 32 ? 1 : 0, QK_LOG2 = 5;
    const int rpg_log2 = walk.waves_log2 + RPW_LOG2, rpg = 1 << rpg_log2;   // rows of a group
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane % LPR, r = lane / LPR;
    // MI355X_EPI_EMIT_Q8_0: the results are also left quantized to Q8_0 for the product that reads them next.  A Q8_0 block is
    // 32 consecutive rows, 2^gpb_log2 groups of this kernel (or a group is whole blocks), so the groups are then dealt in runs (workgroup
    // b: groups b T .. b T + T - 1, T a multiple of those) instead of round-robin, the results of a block meet in LDS and the
    // workgroup rounds them.
    const int gpb_log2 = rpg_log2 < QK_LOG2 ? QK_LOG2 - rpg_log2 : 0, unit_log2 = rpg_log2 < QK_LOG2 ? QK_LOG2 : rpg_log2;
    const bool emit_q8 = (a.e.flags & MI355X_EPI_EMIT_Q8_0) != 0;                          // uniform
    const int group_end = emit_q8 ? min(walk.n_groups, ((int) blockIdx.x + 1) * walk.run) : walk.n_groups;
    __shared__ float q8_rows[NC][W_MAX * RPW < QK ? QK : W_MAX * RPW];
    int group = emit_q8 ? (int) blockIdx.x * walk.run : (int) blockIdx.x;
    const bool idle = emit_q8 && group >= group_end;    // (a grid larger than the runs need: such a workgroup walks one group without storing)
    int64_t row = ((int64_t) group << rpg_log2) + wave * RPW + r;
    bool row_ok = row < a.M && !idle;
    const uint8_t * wrow = (const uint8_t *) a.w + (row_ok ? row : 0) * a.w_nb1;

    // a lane whose block index lies beyond the row reads the row's last block again and counts it with a zero scale
    wraw<T0> blk[NB];
    bool blk_ok[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) blk_ok[b] = j + b * LPR < nbk;
    auto load_blocks = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; ++b) blk[b] = load_wraw<T0>(wrow, blk_ok[b] ? j + b * LPR : nbk - 1);
    };
    // the epilogue operands are fetched early, under the weight stream: lane j of a row stores column j
    float e_bias = 0.0f, e_bcol = 0.0f, e_res = 0.0f;
    auto fetch_epilogue = [&]() __attribute__((always_inline)) {
        if (row_ok && j < NC) {
            if (a.e.flags & MI355X_EPI_BIAS)     e_bias = a.e.bias[row];
            if (a.e.flags & MI355X_EPI_BIAS_COL) e_bcol = a.e.bias[j];
            if (a.e.flags & MI355X_EPI_RESIDUAL) e_res  = *(const float *)(a.e.residual + j * a.d_nb1 + row * 4);
        }
    };
    if (wave < PRO::ROWS) {                             // uniform
        prologue.request();
        __builtin_amdgcn_sched_barrier(0);              // (the scheduler would hoist the weight loads above them again)
        load_blocks();
        if constexpr (PRO::LATE) {
            __builtin_amdgcn_sched_barrier(0);
            prologue.request_late();
        }
        prologue.finish();
    } else {
        load_blocks();
    }
    const char * xbase = prologue.publish(a.x);
    const int32_t * xq   = (const int32_t *) xbase;
    const float *   xd   = (const float *)(xbase + (size_t) NC * K);
    const int32_t * xsum = (const int32_t *)(xbase + (size_t) NC * K + (size_t) NC * nbk * 4);
    int32_t xr[NC][NB][8];
    float   xs[NC][NB];          // scale of the block
    int32_t xo[NC][NB];          // 16 x sum of its quants (Q5_0 weights are stored with an offset of 16)
#pragma unroll
    for (int n = 0; n < NC; ++n) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int kb = j + b * LPR < nbk ? j + b * LPR : 0;
            const int4 x0 = *(const int4 *)(xq + (int64_t) n * (K / 4) + kb * 8), x1 = *(const int4 *)(xq + (int64_t) n * (K / 4) + kb * 8 + 4);
            xr[n][b][0] = x0.x; xr[n][b][1] = x0.y; xr[n][b][2] = x0.z; xr[n][b][3] = x0.w;
            xr[n][b][4] = x1.x; xr[n][b][5] = x1.y; xr[n][b][6] = x1.z; xr[n][b][7] = x1.w;
            xs[n][b] = xd[n * nbk + kb];
            xo[n][b] = T0 == MI355X_TYPE_Q5_0 ? 16 * xsum[n * nbk + kb] : 0;
        }
    }
    fetch_epilogue();

    for (;;) {
        wraw<T0> cur[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) cur[b] = blk[b];
        const int64_t done_row = row;
        const bool done_writer = row_ok && j < NC;
        const float o_bias = e_bias, o_bcol = e_bcol, o_res = e_res;
        // the next row's blocks and epilogue operands travel while this row is worked on
        const int done_group = group;
        group += walk.step;
        const bool more = group < group_end;                // uniform
        if (more) {
            row = ((int64_t) group << rpg_log2) + wave * RPW + r;
            row_ok = row < a.M;
            wrow = (const uint8_t *) a.w + (row_ok ? row : 0) * a.w_nb1;
            load_blocks();
            fetch_epilogue();
        }

        float acc[NC];
#pragma unroll
        for (int n = 0; n < NC; ++n) acc[n] = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            uint32_t q[8];
            const float dw = blk_ok[b] ? h2f((uint16_t) cur[b].d) : 0.0f;
            if constexpr (T0 == MI355X_TYPE_Q8_0) {
#pragma unroll
                for (int i = 0; i < 8; ++i) q[i] = cur[b].q[i];
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    q[i]     = (cur[b].q[i] & 0x0F0F0F0Fu)        | spread4_to_bit4((cur[b].qh >> (4*i))      & 0xFu);
                    q[4 + i] = ((cur[b].q[i] >> 4) & 0x0F0F0F0Fu) | spread4_to_bit4((cur[b].qh >> (16 + 4*i)) & 0xFu);
                }
            }
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                int s = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) s = __builtin_amdgcn_sdot4((int) q[i], xr[n][b][i], s, false);
                if constexpr (T0 == MI355X_TYPE_Q5_0) s -= xo[n][b];
                acc[n] += (float) s * (dw * xs[n][b]);
            }
        }
#pragma unroll
        for (int n = 0; n < NC; ++n) acc[n] = lanes_sum<LPR>(acc[n]);
        // lane j takes column j: one epilogue and one store per lane, and the GELU table's entries of a row come in one trip
        float v = acc[0];
#pragma unroll
        for (int n = 1; n < NC; ++n) v = j == n ? acc[n] : v;
        if (done_writer) {
            v += o_bias + o_bcol;                           // at most one of the two biases is set
            if (a.e.flags & MI355X_EPI_GELU)     v  = gelu_f32(v, a.e.gelu);
            if (a.e.flags & MI355X_EPI_SCALE)    v *= a.e.scale;
            if (a.e.flags & MI355X_EPI_RESIDUAL) v += o_res;
            if (a.e.flags & MI355X_EPI_OUT_F16) *(half_t *)(a.d + j * a.d_nb1 + done_row * 2) = (half_t) v;
            else                                *(float  *)(a.d + j * a.d_nb1 + done_row * 4) = v;
            if (emit_q8) q8_rows[j][(done_group & ((1 << gpb_log2) - 1)) * rpg + wave * RPW + r] = v;
        }
        if (emit_q8 && (((done_group + 1) & ((1 << gpb_log2) - 1)) == 0 || !more)) {          // uniform: blocks of 32 rows are complete (M % 32 == 0)
            // thread (block of the unit, column n, row rr of the block): rounding as quantize_row_q8_0 (ggml-cpu-quants.c:808-865),
            // into the layout of k_quantize_x_q8 for NC rows of M values
            __syncthreads();
            const int u = threadIdx.x >> 5, n = u % NC, rr = threadIdx.x & 31;
            const int64_t bi = ((int64_t)(done_group >> gpb_log2) << (unit_log2 - QK_LOG2)) + u / NC, nb2 = a.M / QK;
            const bool mine = u < NC << (unit_log2 - QK_LOG2);
            const float x = mine ? q8_rows[n][u / NC * QK + rr] : 0.0f;
            const float amax = lanes_max<32>(fabsf(x));
            const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
            const int q = (int) rintf(x * id);
            const int qsum = lanes_sum<32>(q);
            if (mine && !idle && bi < nb2) {
                char * img = (char *) a.e.image;
                ((int8_t *) img)[n * a.M + bi * QK + rr] = (int8_t) q;
                if (rr == 0) {
                    ((float *)(img + (size_t) NC * a.M))[n * nb2 + bi] = h2f(f2h_bits(div127(amax)));
                    ((int32_t *)(img + (size_t) NC * a.M + (size_t) NC * nb2 * 4))[n * nb2 + bi] = qsum;
                }
            }
            __syncthreads();
        }
        if (!more) break;
    }
}

template <int T0, int NC, int LPR, int NB>
__global__ void __launch_bounds__(256) k_gemv_qr(mm_args a, gemv_walk walk) { gemv_qr_rows<T0, NC, LPR, NB, 4>(a, walk); }

// ------------------------------------------------------------------------------------------------------
// Q8_0 weights as tiles for the matrix cores: the product over a matrix long enough to be a stream (the vocabulary
// projection: 70 MB a decode step)
// ------------------------------------------------------------------------------------------------------
// What holds the register kernel back on that matrix is its vector work — 40 v_dot4 per block for five columns — which
// adds to the stream instead of hiding under it.  One v_mfma_i32_16x16x64_i8 takes 16 weight rows x two blocks (the B
// operand: lane (r, g) holds 16 quants of row r — block g / 2 of the pair, half g % 2) against the activations of up
// to eight columns (the A operand, in registers for the whole kernel).  The two blocks of a pair have scales of their
// own, so their sums must not mix: column n sits in A row n with the first block's quants and zeros where the second's
// would be, and in A row 8 + n the other way round.  Result row 4 g' + i then reaches lane (r, g') for the block whose
// scale that lane loads (g' / 2), and what is left per lane and pair of blocks is four conversions, four scale
// products and four f32 fused multiply-adds.  A row's blocks are therefore summed as two interleaved f32 sequences
// (even blocks, odd blocks) that are added at the end.
// Read from the block rows as ggml lays them out, that operand costs more than it saves: every load takes 16 bytes
// from each of 16 rows, at 2-byte alignment, plus a 2-byte load per lane for the scale.  So the matrix is repacked once
// into the order the instruction wants — per 16 rows and pair of blocks, 1024 bytes of quants in lane order followed by
// the 32 scales (68 bytes a row, as before) — and every load of the stream is one aligned, contiguous run of a kilobyte.

__global__ void k_q8_0_tiles_pack(const char * __restrict__ w, int64_t w_nb1, int64_t M, int ksteps, int64_t n_tiles, char * __restrict__ tiles) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;     // (tile, step, lane)
    if (i >= n_tiles * ksteps * 64) return;
    const int lane = (int)(i & 63), r = lane & 15, g = lane >> 4;
    const int64_t ts = i >> 6, tile = ts / ksteps;
    const int step = (int)(ts % ksteps);
    const int64_t row = tile * 16 + r;
    u32x4 q = { 0, 0, 0, 0 };
    uint16_t d = 0;
    if (row < M) {                                     // rows beyond the matrix: zero quants, zero scale
        const char * b = w + row * w_nb1 + (int64_t)(2 * step + (g >> 1)) * 34;
        const u128a2 t = *(const u128a2 *)(b + 2 + 16 * (g & 1));
        q = (u32x4){ t.x, t.y, t.z, t.w };
        d = *(const uint16_t *) b;
    }
    char * o = tiles + ts * Q8T_STEP;
    *(u32x4 *)(o + lane * 16) = q;
    if ((g & 1) == 0) *(uint16_t *)(o + 1024 + ((g >> 1) * 16 + r) * 2) = d;
}

template <int KSTEPS>
static int launch_gemv_q8_0_tiles_k(const mm_args & a, hipStream_t st) {
    const int64_t n_tiles = (a.M + 15) / 16;
    const int64_t resident = 256 * 2 * 4;                 // wavefronts: two workgroups of four per CU
    const int64_t rounds = (n_tiles + resident - 1) / resident;
    const int64_t waves = (n_tiles + rounds - 1) / rounds;
    k_gemv_q8_0_tiles<KSTEPS, false><<<(unsigned)(waves / 4 > 0 ? waves / 4 : 1), 256, 0, st>>>(a, nullptr);
    return launch_status();
}
static bool q8_0_tiles_k_ok(int64_t K) { return K == 384 || K == 512 || K == 768 || K == 1024 || K == 1280; }

// several products over the same activations in one launch (a decode step's Q, K and V): blockIdx.y picks the matrix
struct gemv_group_entry { const char * w; char * d; const float * bias; const char * residual; int64_t d_nb1; int flags; float scale; };
#define GEMV_GROUP_MAX 8
struct gemv_group { gemv_group_entry e[GEMV_GROUP_MAX]; };

template <int T0, int NC, int LPR, int NB>
__global__ void __launch_bounds__(256) k_gemv_qr_group(mm_args a, gemv_walk walk, gemv_group grp) {
    const gemv_group_entry & ge = grp.e[blockIdx.y];
    a.w = ge.w; a.d = ge.d; a.d_nb1 = ge.d_nb1;
    a.e.flags = ge.flags; a.e.scale = ge.scale; a.e.bias = ge.bias; a.e.residual = ge.residual;
    gemv_qr_rows<T0, NC, LPR, NB, 4>(a, walk);
}

// LayerNorm in front of the products, in the same launch.  A decode step's LayerNorm has up to eight rows to work on and is
// over in the latency of a launch; here every workgroup normalizes the rows for itself while its first weight blocks travel —
// the rows in registers between the passes as in k_norm — and leaves them quantized in LDS, where the lanes pick up their
// slices.  The first workgroup also writes what a separate LayerNorm would have left behind: the f32 rows and the Q8_0 form in
// the workspace, for whatever reads them later.
//
// What bounds it is that chain of dependent steps — a memory round trip, two reductions, the block maxima, a barrier, the LDS
// round trip of the quantized rows — about 1 us on top of a launch (1.7 us) when a wavefront has a SIMD to itself, and several
// times that when the workgroups of a CU each run it with the same few wavefronts and pieces of rows that are not there.  Hence
// one workgroup of 8 or 16 wavefronts per CU: the LayerNorm runs once per CU, a row to a wavefront and so at most two on a
// SIMD, on exactly the pieces a row has (JN float4s per lane), and the wavefronts without a row go ahead with the weights.
// Measured, us, with two or three workgroups of four wavefronts to a CU in front (rows x K, columns): 3 x 768 x 768, 3: 7.9 -> 4.5;
// 3072 x 768 to Q8_0, 3: 8.3 -> 6.0; 3 x 1280 x 1280, 5: 8.9 -> 6.5; 5120 x 1280 to Q8_0, 5: 11.2 -> 8.6, 8: 26 -> 9.9;
// 3 x 1024 x 1024, 5: 15.4 -> 5.6 — where the product alone takes 3.7, 6.3, 4.9, 10.1, 11.7 and 4.1.
struct gemv_norm_args {
    const char * src; int64_t src_nb1;
    const float * w; const float * b; float eps;
    char * dst; int64_t dst_nb1;       // f32 rows of the normalized activations
    char * ws;                         // their Q8_0 form (layout of k_quantize_x_q8)
    int threads;                       // of the workgroup
    // EMB instances: row n of the source is not read but made here, token row tok_ids[n] (Q8_0, Q5_0 or F16) plus position row
    // pos_ids[n] (F32) as in k_get_rows_add, and the first workgroup writes it to x0
    const char * tok; int tok_type; int64_t tok_nb1, tok_ne1; const int32_t * tok_ids;
    const char * pos; int64_t pos_nb1, pos_ne1; const int32_t * pos_ids;
    char * x0;
};

// JN: float4s per lane and row, K <= 256 JN (and, for JN = 3, 4, 5, K > 256 (JN - 1): all pieces but the last are whole); W: wavefronts of the workgroup
template <int NC, int JN, int W, bool EMB = false>
struct gemv_norm_prologue {
    const gemv_norm_args & nm; int64_t K; char * lds;
    static constexpr int ROWS = NC < W ? NC : W;
    // wavefront w takes rows w and, where there are more rows than wavefronts, w + W; the rows and the affine vectors are all
    // requested before anything is reduced, so the prologue is one memory round trip long
    static constexpr int RW = (NC + W - 1) / W;             // rows per wavefront
    float4 v[RW][JN], ww[JN], bb[JN];
    // EMB: four values of the token row as they lie in the table (Q8_0: four quants and the block's scale; Q5_0: four bytes
    // of nibbles, the scale and the block's fifth bits; F16: two words) next to the position row's four in v, and whether
    // the row's two indices are inside their tables
    uint32_t tq[EMB ? RW : 1][EMB ? JN : 1], td[EMB ? RW : 1][EMB ? JN : 1], th[EMB ? RW : 1][EMB ? JN : 1];
    int32_t r0[RW], r1[RW];
    bool ok[RW];
    static constexpr bool LATE = EMB;

    // is the lane's piece jj inside the row?
    static __device__ __forceinline__ bool inside(int jj, int lane, int n4) { return (JN >= 3 && JN <= 5 && jj < JN - 1) || lane + jj * WAVE < n4; }

    __device__ __forceinline__ void request() {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int n4 = (int)(K / 4);
        if constexpr (EMB) {                                // the rows' indices now, the rows themselves in request_late()
#pragma unroll
            for (int rr = 0; rr < RW; ++rr) {
                const int row = wave + W * rr < NC ? wave + W * rr : NC - 1;
                r0[rr] = nm.tok_ids[row]; r1[rr] = nm.pos_ids[row];
            }
        }
        // no branch around a load: addresses are clamped into the rows, and a missing affine vector reads the source instead
        const float4 * wp = (const float4 *)(nm.w ? (const char *) nm.w : nm.src), * bp = (const float4 *)(nm.b ? (const char *) nm.b : nm.src);
#pragma unroll
        for (int jj = 0; jj < JN; ++jj) {
            const int c = inside(jj, lane, n4) ? lane + jj * WAVE : n4 - 1;
            if constexpr (!EMB) {
#pragma unroll
                for (int rr = 0; rr < RW; ++rr) {
                    const int row = wave + W * rr < NC ? wave + W * rr : NC - 1;
                    v[rr][jj] = ((const float4 *)(nm.src + row * nm.src_nb1))[c];
                }
            }
            ww[jj] = wp[c]; bb[jj] = bp[c];
        }
    }

    __device__ __forceinline__ void request_late() {
        if constexpr (EMB) {
            const int lane = threadIdx.x & 63;
            const int n4 = (int)(K / 4);
#pragma unroll
            for (int rr = 0; rr < RW; ++rr) {
                ok[rr] = r0[rr] >= 0 && r0[rr] < nm.tok_ne1 && r1[rr] >= 0 && r1[rr] < nm.pos_ne1;
                const uint8_t * tp = (const uint8_t *) nm.tok + (int64_t)(ok[rr] ? r0[rr] : 0) * nm.tok_nb1;
                const float4 *  pp = (const float4 *)(nm.pos + (int64_t)(ok[rr] ? r1[rr] : 0) * nm.pos_nb1);
#pragma unroll
                for (int jj = 0; jj < JN; ++jj) {
                    const int c = inside(jj, lane, n4) ? lane + jj * WAVE : n4 - 1;
                    v[rr][jj] = pp[c];
                    if (nm.tok_type == MI355X_TYPE_Q8_0) {          // uniform
                        const uint8_t * blk = tp + (c >> 3) * 34;
                        td[rr][jj] = ld_u16(blk); tq[rr][jj] = *(const u32a2 *)(blk + 2 + 4 * (c & 7));
                    } else if (nm.tok_type == MI355X_TYPE_Q5_0) {   // (weights j and j + 16 of a block share a byte)
                        const uint8_t * blk = tp + (c >> 3) * 22;
                        td[rr][jj] = ld_u16(blk); th[rr][jj] = *(const u32a2 *)(blk + 2); tq[rr][jj] = *(const u32a2 *)(blk + 6 + 4 * (c & 3));
                    } else {
                        const uint2 h = ((const uint2 *) tp)[c];
                        tq[rr][jj] = h.x; td[rr][jj] = h.y;
                    }
                }
            }
        }
    }

    __device__ __forceinline__ void finish() {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int n4 = (int)(K / 4), nbk = (int)(K / QK);
        const bool writer = blockIdx.x == 0 && blockIdx.y == 0;
        int32_t * xq   = (int32_t *) lds;
        float *   xd   = (float *)(lds + (size_t) NC * K);
        int32_t * xsum = (int32_t *)(lds + (size_t) NC * nbk * 4 + (size_t) NC * K);
#pragma unroll
        for (int rr = 0; rr < RW; ++rr) {
            const int row = wave + W * rr;
            if (row >= NC) break;                           // uniform
            if constexpr (EMB) {                            // the source row: dequantized token values plus position values
#pragma unroll
                for (int jj = 0; jj < JN; ++jj) {
                    float4 e;
                    const uint32_t q = tq[rr][jj], d = td[rr][jj];
                    if (nm.tok_type == MI355X_TYPE_Q8_0) {
                        const float sc = h2f((uint16_t) d);
                        e.x = (float)(int8_t) q * sc;         e.y = (float)(int8_t)(q >> 8) * sc;
                        e.z = (float)(int8_t)(q >> 16) * sc;  e.w = (float)(int8_t)(q >> 24) * sc;
                    } else if (nm.tok_type == MI355X_TYPE_Q5_0) {
                        const float sc = h2f((uint16_t) d);
                        const int c = inside(jj, lane, n4) ? lane + jj * WAVE : n4 - 1;
                        const int j0 = 4 * (c & 7);                                     // first of the lane's four weights in the block
                        const uint32_t nib = (j0 < 16 ? q : q >> 4) & 0x0F0F0F0Fu, hb = th[rr][jj] >> j0;
                        e.x = (float)((int)((nib & 15)         | ((hb & 1) << 4))        - 16) * sc;
                        e.y = (float)((int)(((nib >> 8) & 15)  | (((hb >> 1) & 1) << 4)) - 16) * sc;
                        e.z = (float)((int)(((nib >> 16) & 15) | (((hb >> 2) & 1) << 4)) - 16) * sc;
                        e.w = (float)((int)(((nib >> 24) & 15) | (((hb >> 3) & 1) << 4)) - 16) * sc;
                    } else {
                        e.x = h2f((uint16_t) q); e.y = h2f((uint16_t)(q >> 16)); e.z = h2f((uint16_t) d); e.w = h2f((uint16_t)(d >> 16));
                    }
                    float4 & t = v[rr][jj];
                    const float nan = __builtin_nanf("");
                    t.x = ok[rr] ? e.x + t.x : nan; t.y = ok[rr] ? e.y + t.y : nan; t.z = ok[rr] ? e.z + t.z : nan; t.w = ok[rr] ? e.w + t.w : nan;
                    if (writer && inside(jj, lane, n4)) ((float4 *)(nm.x0 + row * nm.src_nb1))[lane + jj * WAVE] = t;
                }
            }
            float sum = 0.0f;
#pragma unroll
            for (int jj = 0; jj < JN; ++jj) if (inside(jj, lane, n4)) sum += (v[rr][jj].x + v[rr][jj].y) + (v[rr][jj].z + v[rr][jj].w);
            const float mean = wave_sum(sum) / (float) K;
            float sum2 = 0.0f;
#pragma unroll
            for (int jj = 0; jj < JN; ++jj) {
                if (inside(jj, lane, n4)) {
                    float4 & t = v[rr][jj];
                    t.x -= mean; t.y -= mean; t.z -= mean; t.w -= mean;
                    sum2 += (t.x*t.x + t.y*t.y) + (t.z*t.z + t.w*t.w);
                }
            }
            const float scale = 1.0f / sqrtf(wave_sum(sum2) / (float) K + nm.eps);
            // The JN pieces of the row go through each step together — normalize, block maximum, scale, round, block sum, store —
            // and nothing between the steps branches: every piece is a chain of dependent instructions (three cross-lane steps
            // for the maximum, a division, three more for the sum), and side by side the chains fill each other's waits.  (All
            // eight lanes of a block store its scale and its sum: the same value to the same address, instead of a branch
            // around one lane's store.)
            float4 r[JN];
            float amax[JN], id[JN];
            int q[JN][4], qsum[JN];
#pragma unroll
            for (int jj = 0; jj < JN; ++jj) {
                r[jj] = make_float4(v[rr][jj].x * scale, v[rr][jj].y * scale, v[rr][jj].z * scale, v[rr][jj].w * scale);
                {   // (MUL then ADD, two graph nodes: two roundings — without guards around them the two would be contracted)
#pragma clang fp contract(off)
                    if (nm.w) { r[jj].x *= ww[jj].x; r[jj].y *= ww[jj].y; r[jj].z *= ww[jj].z; r[jj].w *= ww[jj].w; }
                    if (nm.b) { r[jj].x += bb[jj].x; r[jj].y += bb[jj].y; r[jj].z += bb[jj].z; r[jj].w += bb[jj].w; }
                }
            }
#pragma unroll
            for (int jj = 0; jj < JN; ++jj)     // (lanes beyond the row hold the clamped last piece: their groups are whole, K % 32 == 0)
                amax[jj] = lanes_max<8>(fmaxf(fmaxf(fabsf(r[jj].x), fabsf(r[jj].y)), fmaxf(fabsf(r[jj].z), fabsf(r[jj].w))));
#pragma unroll
            for (int jj = 0; jj < JN; ++jj) id[jj] = amax[jj] != 0.0f ? 127.0f / amax[jj] : 0.0f;
#pragma unroll
            for (int jj = 0; jj < JN; ++jj) {
                q[jj][0] = (int) rintf(r[jj].x * id[jj]); q[jj][1] = (int) rintf(r[jj].y * id[jj]);
                q[jj][2] = (int) rintf(r[jj].z * id[jj]); q[jj][3] = (int) rintf(r[jj].w * id[jj]);
            }
#pragma unroll
            for (int jj = 0; jj < JN; ++jj) qsum[jj] = lanes_sum<8>((q[jj][0] + q[jj][1]) + (q[jj][2] + q[jj][3]));
#pragma unroll
            for (int jj = 0; jj < JN; ++jj) {
                const int c = lane + jj * WAVE;
                if (inside(jj, lane, n4)) {
                    xq[row * n4 + c] = (q[jj][0] & 0xFF) | ((q[jj][1] & 0xFF) << 8) | ((q[jj][2] & 0xFF) << 16) | ((q[jj][3] & 0xFF) << 24);
                    xd[row * nbk + c / 8] = h2f(f2h_bits(div127(amax[jj])));
                    xsum[row * nbk + c / 8] = qsum[jj];
                }
            }
            if (writer) {
#pragma unroll
                for (int jj = 0; jj < JN; ++jj) if (inside(jj, lane, n4)) ((float4 *)(nm.dst + row * nm.dst_nb1))[lane + jj * WAVE] = r[jj];
            }
        }
    }

    __device__ __forceinline__ const char * publish(const char *) {
        __syncthreads();
        if (blockIdx.x == 0 && blockIdx.y == 0) {           // the workspace copy, 8 bytes per thread and step
            const int pieces = (int)(((size_t) NC * K + (size_t) NC * (K / QK) * 8) / 8);
            for (int i = threadIdx.x; i < pieces; i += nm.threads) ((uint2 *) nm.ws)[i] = ((const uint2 *) lds)[i];
        }
        return lds;
    }
};

template <int T0, int NC, int JN, bool EMB>
__global__ void __launch_bounds__(1024) k_gemv_norm_group(mm_args a, gemv_walk walk, gemv_group grp, gemv_norm_args nm) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const gemv_group_entry & ge = grp.e[blockIdx.y];
    a.w = ge.w; a.d = ge.d; a.d_nb1 = ge.d_nb1;
    a.e.flags = ge.flags; a.e.scale = ge.scale; a.e.bias = ge.bias; a.e.residual = ge.residual;
    gemv_qr_rows<T0, NC, gemv_row_lanes(JN * 8), 1, 16>(a, walk, gemv_norm_prologue<NC, JN, 8, EMB>{ nm, a.K, smem });
}

// the product over the tile-ordered vocabulary matrix with the decoder's last LayerNorm in front, the same way: the
// LayerNorm of the step's rows runs in every workgroup while its first tile row is on the way
template <int KSTEPS, int NC>
__global__ void __launch_bounds__(256, 2) k_gemv_q8_0_tiles_norm(mm_args a, gemv_norm_args nm) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    gemv_q8_0_tiles_body<KSTEPS, false>(a, nullptr, gemv_norm_prologue<NC, (KSTEPS + 3) / 4, 4>{ nm, a.K, smem });
}

template <int KSTEPS, int NC>
static int launch_gemv_q8_0_tiles_norm_kn(const mm_args & a, gemv_norm_args nm, hipStream_t st) {
    const int64_t n_tiles = (a.M + 15) / 16;
    const int64_t resident = 256 * 2 * 4;                 // wavefronts: two workgroups of four per CU
    const int64_t rounds = (n_tiles + resident - 1) / resident;
    const int64_t waves = (n_tiles + rounds - 1) / rounds;
    const unsigned grid = (unsigned)(waves / 4 > 0 ? waves / 4 : 1);
    const size_t lds = (size_t) NC * a.K + (size_t) NC * (a.K / QK) * 8;
    nm.threads = 256;
    k_gemv_q8_0_tiles_norm<KSTEPS, NC><<<grid, 256, lds, st>>>(a, nm);
    return launch_status();
}
template <int KSTEPS>
static int launch_gemv_q8_0_tiles_norm_k(const mm_args & a, const gemv_norm_args & nm, hipStream_t st) {
    switch (a.N) {
        case 1: return launch_gemv_q8_0_tiles_norm_kn<KSTEPS, 1>(a, nm, st);
        case 2: return launch_gemv_q8_0_tiles_norm_kn<KSTEPS, 2>(a, nm, st);
        case 3: return launch_gemv_q8_0_tiles_norm_kn<KSTEPS, 3>(a, nm, st);
        case 4: return launch_gemv_q8_0_tiles_norm_kn<KSTEPS, 4>(a, nm, st);
        case 5: return launch_gemv_q8_0_tiles_norm_kn<KSTEPS, 5>(a, nm, st);
        case 6: return launch_gemv_q8_0_tiles_norm_kn<KSTEPS, 6>(a, nm, st);
        case 7: return launch_gemv_q8_0_tiles_norm_kn<KSTEPS, 7>(a, nm, st);
        case 8: return launch_gemv_q8_0_tiles_norm_kn<KSTEPS, 8>(a, nm, st);
    }
    return MI355X_ERR_INVALID;
}

// ------------------------------------------------------------------------------------------------------
// launches and entry points
// ------------------------------------------------------------------------------------------------------

// Lanes per row of the register kernels, LPR = 16, 32 or 64 with NB <= 3 blocks per lane and N * NB <= 15 block slices of
// activations (120 registers); 0 when the shape does not fit.
//   K <= 2048, up to GEMV_SHORT_ROWS rows in the launch: one block per lane (gemv_row_lanes) — such a product is over in the
//   latency of its loads, and the LayerNorm form, which has the same order of sums, takes what its wavefronts hold at a time.
//   else the fewest lanes per row that still give 512 workgroups: few lanes per row are few idle lanes when the blocks of a row do
//   not divide evenly, and few steps of the sum across lanes; else the most.
static int gemv_r_lanes(int64_t M, int64_t N, int64_t K) {
    const int64_t nbk = K / QK;
    if (nbk <= 64 && M <= GEMV_SHORT_ROWS) return gemv_row_lanes((int) nbk);
    int best = 0;
    for (int lpr = 64; lpr >= 16; lpr /= 2) {
        const int64_t nb = (nbk + lpr - 1) / lpr;
        if (nb > 3 || nb * N > 15) break;
        if (best == 0 || M * lpr / 256 >= 512) best = lpr;
    }
    return best;
}
// bytes of the quantized activations the register variant reads (0: the shape runs with in-kernel quantization)
size_t gemv_ws_bytes(const mi355x_tensor * src0, const mi355x_tensor * src1) {
    const int64_t K = src0->ne[0], N = src1->ne[1];
    if (!gemv_r_lanes(src0->ne[1], N, K)) return 0;
    return round256((size_t)(N * K + N * (K / QK) * 8));
}

// One resident set of workgroups of `waves` wavefronts, each walking its share of the groups of waves * rpw rows: a second, partly
// filled set would double the time.  Returns the grid, 0 for more rows than an int counts.
static unsigned plan_walk(gemv_walk & w, int64_t M, int waves, int rpw, int64_t resident, bool emit_q8) {
    const int rpg = waves * rpw, gpb = rpg < QK ? QK / rpg : 1;
    const int64_t n_groups = (M + rpg - 1) / rpg;
    if (n_groups > 0x3fffffff) return 0;
    const int64_t rounds = (n_groups + resident - 1) / resident, grid = (n_groups + rounds - 1) / rounds;
    w.waves_log2 = waves == 4 ? 2 : waves == 8 ? 3 : 4;
    w.n_groups = (int) n_groups;
    w.run = emit_q8 ? (int)(gpb * ((n_groups + gpb * grid - 1) / (gpb * grid))) : 0;
    w.step = emit_q8 ? 1 : (int) grid;
    return (unsigned) grid;
}

template <int T0, int NC, int LPR, int NB>
static int launch_gemv_r_k(const mm_args & a, hipStream_t st, const gemv_group * grp, int count) {
    const int per_cu = NB > 1 ? 2 : 4;                      // (what the registers allow)
    gemv_walk walk;
    const unsigned grid = plan_walk(walk, a.M, 4, WAVE / LPR, std::max(256 * per_cu / count, 1), ((grp ? grp->e[0].flags : a.e.flags) & MI355X_EPI_EMIT_Q8_0) != 0);
    if (!grid) return MI355X_ERR_UNSUPPORTED;
    if (grp) k_gemv_qr_group<T0, NC, LPR, NB><<<dim3(grid, (unsigned) count), 256, 0, st>>>(a, walk, *grp);
    else     k_gemv_qr<T0, NC, LPR, NB><<<grid, 256, 0, st>>>(a, walk);
    return launch_status();
}
template <int T0, int NC, int LPR>
static int launch_gemv_r_nb(const mm_args & a, int nb, hipStream_t st, const gemv_group * grp, int count) {
    switch (nb) {
        case 1: return launch_gemv_r_k<T0, NC, LPR, 1>(a, st, grp, count);
        case 2: if constexpr (NC * 2 <= 15) return launch_gemv_r_k<T0, NC, LPR, 2>(a, st, grp, count); break;
        case 3: if constexpr (NC * 3 <= 15) return launch_gemv_r_k<T0, NC, LPR, 3>(a, st, grp, count); break;
    }
    return MI355X_ERR_UNSUPPORTED;
}
template <int T0, int NC, int JN>
static int launch_gemv_norm(const mm_args & a, hipStream_t st, const gemv_group & grp, int count, gemv_norm_args nm) {
    // Eight wavefronts to the workgroup while every workgroup then has a CU of its own (a launch of 16 takes 0.5 us longer to get
    // going), 16 from there on (two workgroups on a CU make the rows twice: 7.5 us to 6.5 for 3 x 1280 rows of 1280, 5 columns),
    // and where eight would leave a workgroup several groups to a Q8_0 block of the image.
    const int rpw = WAVE / gemv_row_lanes(JN * 8);
    const bool emit_q8 = (grp.e[0].flags & MI355X_EPI_EMIT_Q8_0) != 0;
    const int waves = (a.M + 8 * rpw - 1) / (8 * rpw) * count <= 256 && (!emit_q8 || 8 * rpw >= QK) ? 8 : 16;
    nm.threads = 64 * waves;
    gemv_walk walk;
    const unsigned grid = plan_walk(walk, a.M, waves, rpw, std::max(256 / count, 1), emit_q8);
    const size_t lds = (size_t) NC * a.K + (size_t) NC * (a.K / QK) * 8;
    if (nm.tok) k_gemv_norm_group<T0, NC, JN, true ><<<dim3(grid, (unsigned) count), 64 * waves, lds, st>>>(a, walk, grp, nm);
    else        k_gemv_norm_group<T0, NC, JN, false><<<dim3(grid, (unsigned) count), 64 * waves, lds, st>>>(a, walk, grp, nm);
    return launch_status();
}
template <int T0, int NC>
static int launch_gemv_r(const mm_args & a, hipStream_t st, const gemv_group * grp, int count, const gemv_norm_args * nm) {
    if (nm) {
        if (a.K <= 512)  return launch_gemv_norm<T0, NC, 2>(a, st, *grp, count, *nm);
        if (a.K <= 768)  return launch_gemv_norm<T0, NC, 3>(a, st, *grp, count, *nm);
        if (a.K <= 1024) return launch_gemv_norm<T0, NC, 4>(a, st, *grp, count, *nm);
        if (a.K <= 1280) return launch_gemv_norm<T0, NC, 5>(a, st, *grp, count, *nm);
        return launch_gemv_norm<T0, NC, 8>(a, st, *grp, count, *nm);
    }
    int lpr = gemv_r_lanes(a.M * count, NC, a.K);
    if (!lpr) return MI355X_ERR_UNSUPPORTED;
    // with the Q8_0 emission a workgroup owns whole blocks of 32 rows, so there are M / 32 workgroups at most: the fewer lanes a
    // row takes, the fewer groups each of them walks one after the other
    const bool emit_q8 = ((grp ? grp->e[0].flags : a.e.flags) & MI355X_EPI_EMIT_Q8_0) != 0;
    if (emit_q8 && a.M > GEMV_SHORT_ROWS && (a.K / QK + 15) / 16 <= 3 && (a.K / QK + 15) / 16 * NC <= 15) lpr = 16;
    const int nb = (int)((a.K / QK + lpr - 1) / lpr);
    switch (lpr) {
        case 16: return launch_gemv_r_nb<T0, NC, 16>(a, nb, st, grp, count);
        case 32: return launch_gemv_r_nb<T0, NC, 32>(a, nb, st, grp, count);
        default: return launch_gemv_r_nb<T0, NC, 64>(a, nb, st, grp, count);
    }
}
template <int T0>
static int launch_gemv_r_n(const mm_args & a, hipStream_t st, const gemv_group * grp = nullptr, int count = 1, const gemv_norm_args * nm = nullptr) {
    switch (a.N) {
        case 1: return launch_gemv_r<T0, 1>(a, st, grp, count, nm);
        case 2: return launch_gemv_r<T0, 2>(a, st, grp, count, nm);
        case 3: return launch_gemv_r<T0, 3>(a, st, grp, count, nm);
        case 4: return launch_gemv_r<T0, 4>(a, st, grp, count, nm);
        case 5: return launch_gemv_r<T0, 5>(a, st, grp, count, nm);
        case 6: return launch_gemv_r<T0, 6>(a, st, grp, count, nm);
        case 7: return launch_gemv_r<T0, 7>(a, st, grp, count, nm);
        case 8: return launch_gemv_r<T0, 8>(a, st, grp, count, nm);
    }
    return MI355X_ERR_INVALID;
}

template <int T0, int NC>
static int launch_gemv(const mm_args & a, hipStream_t st) {
    const size_t lds = (size_t) NC * a.K + (size_t) NC * (a.K / QK) * 8;
    // lanes per row: the smallest split of a row's blocks that still yields enough workgroups to fill 256 CUs
    int lpr = 8;
    while (lpr < 64 && a.M * lpr / 256 < 512) lpr *= 2;
    const int rows_per_wg = 4 * (WAVE / lpr);
    // a workgroup walks several row groups when there are more than three per CU, so that the activations are quantized
    // fewer times; the groups are dealt out evenly
    const int64_t n_groups = (a.M + rows_per_wg - 1) / rows_per_wg;
    const int64_t rounds   = (n_groups + 767) / 768;
    const unsigned grid    = (unsigned)((n_groups + rounds - 1) / rounds);
    switch (lpr) {
        case 8:  k_gemv_q<T0, NC, 8 ><<<grid, 256, lds, st>>>(a); break;
        case 16: k_gemv_q<T0, NC, 16><<<grid, 256, lds, st>>>(a); break;
        case 32: k_gemv_q<T0, NC, 32><<<grid, 256, lds, st>>>(a); break;
        default: k_gemv_q<T0, NC, 64><<<grid, 256, lds, st>>>(a); break;
    }
    return launch_status();
}

template <int T0>
static int launch_gemv_n(const mm_args & a, hipStream_t st) {
    switch (a.N) {
        case 1: return launch_gemv<T0, 1>(a, st);
        case 2: return launch_gemv<T0, 2>(a, st);
        case 3: return launch_gemv<T0, 3>(a, st);
        case 4: return launch_gemv<T0, 4>(a, st);
        case 5: return launch_gemv<T0, 5>(a, st);
        case 6: return launch_gemv<T0, 6>(a, st);
        case 7: return launch_gemv<T0, 7>(a, st);
        case 8: return launch_gemv<T0, 8>(a, st);
    }
    return MI355X_ERR_INVALID;
}
int launch_quantize_x_q8(const char * x, int64_t x_nb1, int64_t K, int64_t N, char * ws, hipStream_t st) {
    k_quantize_x_q8<<<(unsigned)((N * (K / 4) + 255) / 256), 256, 0, st>>>(x, x_nb1, K, N, ws);
    return launch_status();
}
int launch_gemv_ws(int type, const mm_args & a, hipStream_t st) {
    return type == MI355X_TYPE_Q8_0 ? launch_gemv_r_n<MI355X_TYPE_Q8_0>(a, st) : launch_gemv_r_n<MI355X_TYPE_Q5_0>(a, st);
}
int launch_gemv_lds(int type, const mm_args & a, hipStream_t st) {
    return type == MI355X_TYPE_Q8_0 ? launch_gemv_n<MI355X_TYPE_Q8_0>(a, st) : launch_gemv_n<MI355X_TYPE_Q5_0>(a, st);
}

// a LayerNorm in front of the products: what the kernels take, and the tensors for the case that it gets a launch of its own
struct gemv_norm_source {
    gemv_norm_args nm;
    const mi355x_tensor * src, * normed;
    const mi355x_tensor * tok, * tok_ids, * pos, * pos_ids;    // of the gathering form, else NULL
};

// the few-column form of mi355x_mul_mat_group: quantized weights of one type and shape, activations quantized once
static int group_gemv(const mi355x_mul_mat_item * items, int count, const mi355x_tensor * src1, int flags,
                              void * workspace, size_t workspace_size, void * stream, gemv_norm_source * ns) {
    const mi355x_tensor * w0 = items[0].src0;
    if (count > GEMV_GROUP_MAX || src1->type != MI355X_TYPE_F32 || mm_path(w0, src1) != MM_GEMV) return MI355X_ERR_UNSUPPORTED;
    if (w0->type != MI355X_TYPE_Q8_0 && w0->type != MI355X_TYPE_Q5_0) return MI355X_ERR_UNSUPPORTED;
    mm_args a;
    a.K = w0->ne[0]; a.M = w0->ne[1]; a.N = src1->ne[1];
    if (src1->ne[0] != a.K || a.K % QK != 0) return MI355X_ERR_INVALID;
    if (a.M == 0 || a.N == 0) return MI355X_OK;
    const size_t need = gemv_ws_bytes(w0, src1);
    if (!need || !gemv_r_lanes(a.M * count, a.N, a.K)) return MI355X_ERR_UNSUPPORTED;
    if (!workspace || workspace_size < need || (uintptr_t) workspace % 16 != 0) return MI355X_ERR_WORKSPACE;
    gemv_group grp;
    bool any_gelu = false;
    for (int i = 0; i < count; ++i) {
        const mi355x_tensor * w = items[i].src0, * d = items[i].dst;
        const mi355x_epilogue * e = items[i].epi;
        if (!w || !d) return MI355X_ERR_INVALID;
        if (w->type != w0->type || w->ne[0] != a.K || w->ne[1] != a.M || w->ne[2] != 1 || w->ne[3] != 1 || w->nb[1] != w0->nb[1] || (uintptr_t) w->data % 2 != 0) return MI355X_ERR_UNSUPPORTED;
        if (e && (e->flags & MI355X_EPI_EMIT_F16)) return MI355X_ERR_UNSUPPORTED;
        int ef = e ? (e->flags & 63) : 0;
        const int td = (ef & MI355X_EPI_OUT_F16) ? MI355X_TYPE_F16 : MI355X_TYPE_F32;
        if (d->type != td || d->ne[0] != a.M || d->ne[1] != a.N || d->ne[2] != 1 || d->ne[3] != 1 || d->nb[0] != type_size(td)) return MI355X_ERR_UNSUPPORTED;
        if ((ef & (MI355X_EPI_BIAS | MI355X_EPI_BIAS_COL)) && !e->bias) return MI355X_ERR_INVALID;
        if ((ef & MI355X_EPI_BIAS) && (ef & MI355X_EPI_BIAS_COL)) return MI355X_ERR_INVALID;
        if ((ef & MI355X_EPI_RESIDUAL) && (!e->residual || (ef & MI355X_EPI_OUT_F16))) return MI355X_ERR_INVALID;
        if (e && (e->flags & MI355X_EPI_EMIT_Q8_0)) {           // the result also as Q8_0: one product per launch, whole blocks
            if (count != 1 || (ef & MI355X_EPI_OUT_F16) || a.M % QK != 0) return MI355X_ERR_UNSUPPORTED;
            if (!e->image || (uintptr_t) e->image % 16 != 0) return MI355X_ERR_INVALID;
            ef |= MI355X_EPI_EMIT_Q8_0;
        }
        any_gelu = any_gelu || (ef & MI355X_EPI_GELU);
        grp.e[i] = { (const char *) w->data, (char *) d->data, e ? (const float *) e->bias : nullptr, e ? (const char *) e->residual : nullptr, (int64_t) d->nb[1], ef, e ? e->scale : 1.0f };
    }
    a.w = (const char *) w0->data; a.x = (const char *) src1->data; a.d = (char *) items[0].dst->data;
    a.w_nb1 = w0->nb[1]; a.w_nb2 = a.w_nb3 = 0;
    a.x_nb1 = src1->nb[1]; a.x_nb2 = a.x_nb3 = 0;
    a.d_nb1 = items[0].dst->nb[1]; a.d_nb2 = a.d_nb3 = 0;
    a.ne12 = a.ne13 = a.r2 = a.r3 = 1;
    a.e.flags = 0; a.e.scale = 1.0f; a.e.bias = nullptr; a.e.residual = nullptr; a.e.gelu = nullptr;
    a.e.image = (grp.e[0].flags & MI355X_EPI_EMIT_Q8_0) ? (half_t *) items[0].epi->image : nullptr;
    if (any_gelu && !(a.e.gelu = gelu_table_device())) return MI355X_ERR_HIP;
    hipStream_t st = (hipStream_t) stream;
    if (ns) {                                               // the LayerNorm in front: it writes src1 and the workspace
        ns->nm.ws = (char *) workspace;
        if (a.M * count <= GEMV_SHORT_ROWS)                 // ... in the same launch
            return w0->type == MI355X_TYPE_Q8_0 ? launch_gemv_r_n<MI355X_TYPE_Q8_0>(a, st, &grp, count, &ns->nm) : launch_gemv_r_n<MI355X_TYPE_Q5_0>(a, st, &grp, count, &ns->nm);
        // a long stream of weights: a launch more is nothing beside it, and the LayerNorm's registers would cost it wavefronts
        if (ns->tok) if (const int rc = mi355x_get_rows_add(ns->tok, ns->tok_ids, ns->pos, ns->pos_ids, ns->src, stream)) return rc;
        if (const int rc = mi355x_norm_emit_q8_0(ns->src, ns->normed, ns->nm.eps, ns->nm.w, ns->nm.b, workspace, stream)) return rc;
        flags |= MI355X_MM_WS_READY;
    }
    if (!(flags & MI355X_MM_WS_READY)) {
        k_quantize_x_q8<<<(unsigned)((a.N * (a.K / 4) + 255) / 256), 256, 0, st>>>(a.x, a.x_nb1, a.K, a.N, (char *) workspace);
        if (const int rc = launch_status()) return rc;
    }
    if (flags & MI355X_MM_PREPARE_ONLY) return MI355X_OK;
    a.x = (const char *) workspace;
    return w0->type == MI355X_TYPE_Q8_0 ? launch_gemv_r_n<MI355X_TYPE_Q8_0>(a, st, &grp, count) : launch_gemv_r_n<MI355X_TYPE_Q5_0>(a, st, &grp, count);
}

int mul_mat_group_gemv(const mi355x_mul_mat_item * items, int count, const mi355x_tensor * src1, int flags, void * workspace, size_t workspace_size, void * stream) {
    return group_gemv(items, count, src1, flags, workspace, workspace_size, stream, nullptr);
}

// the checks common to the LayerNorm-and-products entries; `nm` arrives with the gather fields set or zero
static int norm_mul_mat_group(const mi355x_tensor * src, const mi355x_tensor * normed, float eps, const float * w, const float * b,
                              const mi355x_mul_mat_item * items, int count, void * workspace, size_t workspace_size, void * stream, gemv_norm_source ns) {
    if (!src || !normed || !items || count < 1 || !(eps >= 0.0f)) return MI355X_ERR_INVALID;
    if (!items[0].src0 || !items[0].dst) return MI355X_ERR_INVALID;
    if (src->type != MI355X_TYPE_F32 || normed->type != MI355X_TYPE_F32 || src->nb[0] != 4 || normed->nb[0] != 4) return MI355X_ERR_UNSUPPORTED;
    for (int i = 0; i < 4; ++i) if (src->ne[i] != normed->ne[i]) return MI355X_ERR_INVALID;
    const int64_t K = src->ne[0], N = src->ne[1];
    if (src->ne[2] != 1 || src->ne[3] != 1 || N < 1 || N > MI355X_GEMV_MAX_COLS || K % QK != 0 || K > 2048) return MI355X_ERR_UNSUPPORTED;
    if (!aligned16(src) || !aligned16(normed) || (uintptr_t) w % 16 != 0 || (uintptr_t) b % 16 != 0) return MI355X_ERR_UNSUPPORTED;
    if (blck_size(items[0].src0->type) <= 1) return MI355X_ERR_UNSUPPORTED;
    gemv_norm_args & nm = ns.nm;
    nm.src = (const char *) src->data; nm.src_nb1 = (int64_t) src->nb[1]; nm.w = w; nm.b = b; nm.eps = eps;
    nm.dst = (char *) normed->data; nm.dst_nb1 = (int64_t) normed->nb[1]; nm.ws = nullptr;
    ns.src = src; ns.normed = normed;
    return group_gemv(items, count, normed, 0, workspace, workspace_size, stream, &ns);
}

extern "C" int mi355x_norm_mul_mat_group(const mi355x_tensor * src, const mi355x_tensor * normed, float eps, const float * w, const float * b,
                                         const mi355x_mul_mat_item * items, int count, void * workspace, size_t workspace_size, void * stream) {
    return norm_mul_mat_group(src, normed, eps, w, b, items, count, workspace, workspace_size, stream, gemv_norm_source{});
}

extern "C" int mi355x_embed_norm_mul_mat_group(const mi355x_tensor * tok, const mi355x_tensor * tok_ids, const mi355x_tensor * pos, const mi355x_tensor * pos_ids,
                                               const mi355x_tensor * x0, const mi355x_tensor * normed, float eps, const float * w, const float * b,
                                               const mi355x_mul_mat_item * items, int count, void * workspace, size_t workspace_size, void * stream) {
    if (!tok || !tok_ids || !pos || !pos_ids || !x0) return MI355X_ERR_INVALID;
    if (tok_ids->type != MI355X_TYPE_I32 || pos_ids->type != MI355X_TYPE_I32 || pos->type != MI355X_TYPE_F32) return MI355X_ERR_UNSUPPORTED;
    if (tok->type != MI355X_TYPE_Q8_0 && tok->type != MI355X_TYPE_Q5_0 && tok->type != MI355X_TYPE_F16) return MI355X_ERR_UNSUPPORTED;
    const int64_t K = x0->ne[0], N = x0->ne[1];
    for (int i = 1; i < 4; ++i) if (tok_ids->ne[i] != 1 || pos_ids->ne[i] != 1) return MI355X_ERR_UNSUPPORTED;
    if (tok_ids->ne[0] != N || pos_ids->ne[0] != N || tok_ids->nb[0] != 4 || pos_ids->nb[0] != 4) return MI355X_ERR_UNSUPPORTED;
    if (tok->ne[2] != 1 || tok->ne[3] != 1 || pos->ne[2] != 1 || pos->ne[3] != 1) return MI355X_ERR_UNSUPPORTED;
    if (tok->ne[0] != K || pos->ne[0] != K || pos->nb[0] != 4 || tok->nb[0] != type_size(tok->type)) return MI355X_ERR_INVALID;
    // (a lane reads four values of a row at a time: 8 bytes of an F16 row, 16 of a position row; quantized blocks sit at even addresses)
    const uintptr_t ta = tok->type == MI355X_TYPE_F16 ? 8 : 2;
    if ((uintptr_t) tok->data % ta != 0 || tok->nb[1] % ta != 0 || (uintptr_t) pos->data % 16 != 0 || pos->nb[1] % 16 != 0 ||
        (uintptr_t) tok_ids->data % 4 != 0 || (uintptr_t) pos_ids->data % 4 != 0) return MI355X_ERR_UNSUPPORTED;
    gemv_norm_source ns{};
    ns.tok = tok; ns.tok_ids = tok_ids; ns.pos = pos; ns.pos_ids = pos_ids;
    gemv_norm_args & nm = ns.nm;
    nm.tok = (const char *) tok->data; nm.tok_type = tok->type; nm.tok_nb1 = (int64_t) tok->nb[1]; nm.tok_ne1 = tok->ne[1]; nm.tok_ids = (const int32_t *) tok_ids->data;
    nm.pos = (const char *) pos->data; nm.pos_nb1 = (int64_t) pos->nb[1]; nm.pos_ne1 = pos->ne[1]; nm.pos_ids = (const int32_t *) pos_ids->data;
    nm.x0 = (char *) x0->data;
    return norm_mul_mat_group(x0, normed, eps, w, b, items, count, workspace, workspace_size, stream, ns);
}
extern "C" size_t mi355x_q8_0_tiles_size(int64_t K, int64_t M) {
    if (K <= 0 || M <= 0 || K % 64 != 0) return 0;
    return (size_t)((M + 15) / 16) * (size_t)(K / 64) * Q8T_STEP;
}

extern "C" int mi355x_q8_0_tiles_pack(const mi355x_tensor * src0, void * tiles, void * stream) {
    if (!src0 || !tiles) return MI355X_ERR_INVALID;
    if (src0->type != MI355X_TYPE_Q8_0 || src0->ne[2] != 1 || src0->ne[3] != 1 || src0->nb[0] != 34) return MI355X_ERR_UNSUPPORTED;
    const int64_t K = src0->ne[0], M = src0->ne[1];
    if (K <= 0 || M <= 0 || K % 64 != 0 || (uintptr_t) src0->data % 2 != 0 || src0->nb[1] % 2 != 0 || (uintptr_t) tiles % 16 != 0) return MI355X_ERR_UNSUPPORTED;
    const int64_t n_tiles = (M + 15) / 16, threads = n_tiles * (K / 64) * 64;
    if ((threads + 255) / 256 > 0x7fffffff) return MI355X_ERR_UNSUPPORTED;
    k_q8_0_tiles_pack<<<(unsigned)((threads + 255) / 256), 256, 0, (hipStream_t) stream>>>((const char *) src0->data, (int64_t) src0->nb[1], M, (int)(K / 64), n_tiles, (char *) tiles);
    return launch_status();
}

extern "C" int mi355x_mul_mat_q8_0_tiles(const void * tiles, int64_t K, int64_t M, const mi355x_tensor * src1, const mi355x_tensor * dst,
                                         int flags, void * workspace, size_t workspace_size, void * stream) {
    if (!tiles || !src1 || !dst) return MI355X_ERR_INVALID;
    if (!q8_0_tiles_k_ok(K) || M <= 0 || (uintptr_t) tiles % 16 != 0) return MI355X_ERR_UNSUPPORTED;
    if (flags & ~(MI355X_EPI_OUT_F16 | MI355X_MM_WS_READY | MI355X_MM_PREPARE_ONLY)) return MI355X_ERR_UNSUPPORTED;
    const int td = (flags & MI355X_EPI_OUT_F16) ? MI355X_TYPE_F16 : MI355X_TYPE_F32;
    const int64_t N = src1->ne[1];
    if (src1->type != MI355X_TYPE_F32 || dst->type != td || src1->nb[0] != 4 || dst->nb[0] != type_size(td)) return MI355X_ERR_UNSUPPORTED;
    if (src1->ne[0] != K || dst->ne[0] != M || dst->ne[1] != N) return MI355X_ERR_INVALID;
    if (N < 1 || N > MI355X_GEMV_MAX_COLS || src1->ne[2] != 1 || src1->ne[3] != 1 || dst->ne[2] != 1 || dst->ne[3] != 1 || !aligned16(src1)) return MI355X_ERR_UNSUPPORTED;
    const size_t need = round256((size_t)(N * K + N * (K / QK) * 8));
    if (!workspace || workspace_size < need || (uintptr_t) workspace % 16 != 0) return MI355X_ERR_WORKSPACE;
    hipStream_t st = (hipStream_t) stream;
    if (!(flags & MI355X_MM_WS_READY)) {
        k_quantize_x_q8<<<(unsigned)((N * (K / 4) + 255) / 256), 256, 0, st>>>((const char *) src1->data, (int64_t) src1->nb[1], K, N, (char *) workspace);
        if (const int rc = launch_status()) return rc;
    }
    if (flags & MI355X_MM_PREPARE_ONLY) return MI355X_OK;
    mm_args a;
    a.K = K; a.M = M; a.N = N;
    a.w = (const char *) tiles; a.x = (const char *) workspace; a.d = (char *) dst->data;
    a.w_nb1 = a.w_nb2 = a.w_nb3 = 0; a.x_nb1 = a.x_nb2 = a.x_nb3 = 0;
    a.d_nb1 = dst->nb[1]; a.d_nb2 = a.d_nb3 = 0;
    a.ne12 = a.ne13 = a.r2 = a.r3 = 1;
    a.e.flags = flags & MI355X_EPI_OUT_F16; a.e.scale = 1.0f; a.e.bias = nullptr; a.e.residual = nullptr; a.e.gelu = nullptr; a.e.image = nullptr;
    switch (K) {
        case 384:  return launch_gemv_q8_0_tiles_k<6>(a, st);
        case 512:  return launch_gemv_q8_0_tiles_k<8>(a, st);
        case 768:  return launch_gemv_q8_0_tiles_k<12>(a, st);
        case 1024: return launch_gemv_q8_0_tiles_k<16>(a, st);
        default:   return launch_gemv_q8_0_tiles_k<20>(a, st);
    }
}

extern "C" int mi355x_norm_mul_mat_q8_0_tiles(const void * tiles, int64_t K, int64_t M, const mi355x_tensor * src, const mi355x_tensor * normed,
                                              float eps, const float * w, const float * b, const mi355x_tensor * dst, int flags,
                                              void * workspace, size_t workspace_size, void * stream) {
    if (!tiles || !src || !normed || !dst || !(eps >= 0.0f)) return MI355X_ERR_INVALID;
    if (!q8_0_tiles_k_ok(K) || M <= 0 || (uintptr_t) tiles % 16 != 0) return MI355X_ERR_UNSUPPORTED;
    if (flags & ~MI355X_EPI_OUT_F16) return MI355X_ERR_UNSUPPORTED;
    const int td = (flags & MI355X_EPI_OUT_F16) ? MI355X_TYPE_F16 : MI355X_TYPE_F32;
    const int64_t N = src->ne[1];
    if (src->type != MI355X_TYPE_F32 || normed->type != MI355X_TYPE_F32 || dst->type != td || src->nb[0] != 4 || normed->nb[0] != 4 || dst->nb[0] != type_size(td)) return MI355X_ERR_UNSUPPORTED;
    for (int i = 0; i < 4; ++i) if (src->ne[i] != normed->ne[i]) return MI355X_ERR_INVALID;
    if (src->ne[0] != K || dst->ne[0] != M || dst->ne[1] != N) return MI355X_ERR_INVALID;
    if (N < 1 || N > MI355X_GEMV_MAX_COLS || src->ne[2] != 1 || src->ne[3] != 1 || dst->ne[2] != 1 || dst->ne[3] != 1) return MI355X_ERR_UNSUPPORTED;
    if (!aligned16(src) || !aligned16(normed) || (uintptr_t) w % 16 != 0 || (uintptr_t) b % 16 != 0) return MI355X_ERR_UNSUPPORTED;
    const size_t need = round256((size_t)(N * K + N * (K / QK) * 8));
    if (!workspace || workspace_size < need || (uintptr_t) workspace % 16 != 0) return MI355X_ERR_WORKSPACE;
    gemv_norm_args nm{};
    nm.src = (const char *) src->data; nm.src_nb1 = (int64_t) src->nb[1]; nm.w = w; nm.b = b; nm.eps = eps;
    nm.dst = (char *) normed->data; nm.dst_nb1 = (int64_t) normed->nb[1]; nm.ws = (char *) workspace;
    mm_args a;
    a.K = K; a.M = M; a.N = N;
    a.w = (const char *) tiles; a.x = (const char *) workspace; a.d = (char *) dst->data;
    a.w_nb1 = a.w_nb2 = a.w_nb3 = 0; a.x_nb1 = a.x_nb2 = a.x_nb3 = 0;
    a.d_nb1 = dst->nb[1]; a.d_nb2 = a.d_nb3 = 0;
    a.ne12 = a.ne13 = a.r2 = a.r3 = 1;
    a.e.flags = flags & MI355X_EPI_OUT_F16; a.e.scale = 1.0f; a.e.bias = nullptr; a.e.residual = nullptr; a.e.gelu = nullptr; a.e.image = nullptr;
    hipStream_t st = (hipStream_t) stream;
    switch (K) {
        case 384:  return launch_gemv_q8_0_tiles_norm_k<6>(a, nm, st);
        case 512:  return launch_gemv_q8_0_tiles_norm_k<8>(a, nm, st);
        case 768:  return launch_gemv_q8_0_tiles_norm_k<12>(a, nm, st);
        case 1024: return launch_gemv_q8_0_tiles_norm_k<16>(a, nm, st);
        default:   return launch_gemv_q8_0_tiles_norm_k<20>(a, nm, st);
    }
}
