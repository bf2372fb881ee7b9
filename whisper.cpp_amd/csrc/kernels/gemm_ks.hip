// MUL_MAT over f16 weights for problems too small to fill the device with 128-wide tiles, for a handful of columns, and for
// operands whose rows are not 16-byte aligned: k_gemm_ks.
//
// What bounds such a product is not the matrix cores but the time until the first operands are there and how much of the
// device asks for them: a decoder's 1280 x 1280 product over 5 columns is 20 tiles of 64 x 64 with 20 dependent K steps each,
// 10.3 us where its 3.3 MB of weights need 1.  Here tiles are small and the K range of a tile is dealt to the KW wavefronts of
// a workgroup (units of 64 values, round robin: the wavefronts together read consecutive 128-byte lines).  No operand is used
// by two wavefronts, so each streams its own and the K loop has no barrier; the partial tiles meet once, in LDS, where the
// epilogue reads them.  k_gemm_ks streams through LDS, k_gemm_kd (any alignment, any K) straight into registers.
//
// The weights are the A operand of v_mfma_f32_16x16x32_f16, the activations (src1) the B operand: lane l holds row / column
// l % 16 and k = 8 (l / 16) .. + 7 of a 32-deep step, and the result's registers are 4 consecutive m of one dst row.
// Rows past M and columns past N are read from the last valid one and not stored; a K that is no multiple of 64 ends in one
// unit whose loads are guarded value by value.
#include "gemm_ks.h"

#include <atomic>

#define KS_UNIT 64

template <int N>
__device__ __forceinline__ void ks_wait_vmcnt() {             // s_waitcnt vmcnt(N) only; what is read from LDS stays behind it
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

typedef float ks_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef half_t ks_h8 __attribute__((ext_vector_type(8), aligned(2)));
typedef half_t ks_h4 __attribute__((ext_vector_type(4), aligned(2)));

template <int MT, int NT, int KW> constexpr size_t ks_red_bytes() { return (size_t) KW * 16 * NT * (16 * MT + 4) * sizeof(float); }

// the epilogue of four consecutive m of a column, and their way out (EMIT: a column past N or rows past M only pass through)
template <bool EMIT>
__device__ __forceinline__ void ks_store4(float4_t & v, int64_t m, int64_t n, const mm_args & a, char * db, const epi_args & epi, int64_t batch_off, int64_t d_nb1) {
    const bool row = n < a.N;
    if (m + 3 < a.M) {
        const int64_t nc = row ? n : a.N - 1;
        if (epi.flags & MI355X_EPI_BIAS) v += *(const ks_f4 *)(epi.bias + m);
        if (epi.flags & MI355X_EPI_BIAS_COL) v += epi.bias[nc];
        if (epi.flags & MI355X_EPI_GELU) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gelu_f32(v[e], epi.gelu);
        }
        if (epi.flags & MI355X_EPI_SCALE) v *= epi.scale;
        if (epi.flags & MI355X_EPI_RESIDUAL) v += *(const ks_f4 *)(epi.residual + batch_off + nc * d_nb1 + m * 4);
        if (row) {
            if (epi.flags & MI355X_EPI_OUT_F16) *(ks_h4 *)(db + n * d_nb1 + m * 2) = (ks_h4){ (half_t) v[0], (half_t) v[1], (half_t) v[2], (half_t) v[3] };
            else if (!EMIT || !(epi.flags & MI355X_EPI_IMAGE_ONLY)) *(ks_f4 *)(db + n * d_nb1 + m * 4) = v;
        }
    } else if (row && m < a.M) {
        for (int e = 0; e < 4 && m + e < a.M; ++e) {
            const float y = apply_epilogue(v[e], epi, m + e, n, batch_off + n * d_nb1 + (m + e) * 4);
            if (epi.flags & MI355X_EPI_OUT_F16) *(half_t *)(db + n * d_nb1 + (m + e) * 2) = (half_t) y;
            else                                *(float  *)(db + n * d_nb1 + (m + e) * 4) = y;
        }
    }
}

// The partial tiles of the KW wavefronts meet in `red` ([KW][16 NT][LD] floats, free when every wavefront is past its loop) and
// leave through the epilogue.  EMIT: MI355X_EPI_EMIT_F16 (a block of 32 m is 8 consecutive lanes).
template <int MT, int NT, int KW, bool EMIT, int H = 1>
__device__ __forceinline__ void ks_finish(float4_t (&acc)[MT][NT], float * red, const mm_args & a, char * db, const epi_args & epi, int64_t batch_off,
                                          int64_t d_nb1, int64_t m0, int64_t n0) {
    static_assert(!EMIT || MT % 2 == 0, "whole Q8_0 blocks per tile");
    constexpr int LD = 16 * MT + 4;                     // (+ 4: the 16 rows n of a result register start 4 banks apart)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, q = lane >> 4;
    // result register e of a 16x16 tile: column (n) lane % 16, row (m) 4 (lane / 16) + e
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) *(float4_t *)(red + (wave * 16 * NT + 16 * j + r16) * LD + 16 * i + 4 * q) = acc[i][j];
    __syncthreads();
    constexpr int MR = 16 * MT / H, NR = 16 * NT / H;   // rows and columns of the tile
    constexpr int PIECES = NR * MR / 4;                 // (n, four consecutive m)
#pragma unroll
    for (int p0 = 0; p0 < PIECES; p0 += 64 * KW) {
        const int p = p0 + tid;
        if (PIECES % (64 * KW) != 0 && p >= PIECES) break;
        const int nl = p / (MR / 4), ml = p % (MR / 4) * 4;
        float4_t v = *(const float4_t *)(red + nl * LD + ml);
#pragma unroll
        for (int w = 0; w < KW; ++w)
#pragma unroll
            for (int h = 0; h < H; ++h) if (w + h > 0) v += *(const float4_t *)(red + (w * 16 * NT + nl + h * NR) * LD + ml + h * MR);
        const int64_t n = n0 + nl, m = m0 + ml;
        const bool row = n < a.N, whole = m + 3 < a.M;
        if (!EMIT && (!row || m >= a.M)) continue;
        ks_store4<EMIT>(v, m, n, a, db, epi, batch_off, d_nb1);
        if (EMIT) {                                     // M is a multiple of 32: a block of 8 lanes is inside dst or outside
            float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
            amax = lanes_max<8>(amax);
            const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
            const float dq = h2f(f2h_bits(div127(amax)));
            if (row && whole)
                *(half4_t *)(epi.image + n * a.M + m) = (half4_t){ (half_t)((rintf(v[0] * id) + 0.0f) * dq), (half_t)((rintf(v[1] * id) + 0.0f) * dq),
                                                                   (half_t)((rintf(v[2] * id) + 0.0f) * dq), (half_t)((rintf(v[3] * id) + 0.0f) * dq) };
        }
    }
}

// The same with the operands streamed through LDS: rows at 16-byte alignment, K a multiple of 64.  A fragment load straight
// from global memory takes 16 rows in every 16 lanes, 16 cache lines where 16 consecutive lanes could share two, and the
// L1 cache looks up one line a clock: 16 B per clock and CU.  global_load_lds reads 8 whole 128-byte row pieces instead, and
// the fragments come out of LDS.  Every wavefront streams its own units through its own D buffers, so the loop has no
// barrier in it.
// LDS layout of f16 rows: row pairs form 256-byte lines, the 16-byte chunk c of row r sits in slot (r & 1) * 8 + (c ^ (line & 7))
// of line r / 2 (the 16 rows of a fragment read then cover all banks once); f32 rows are one line each, chunk c in slot c ^ (r & 15).
// XR: rows of src1 that are loaded (8 with at most 8 columns: the other columns of the result are not stored).
// H = 2, at most 8 columns: the tile is 8 rows, and the 16 rows and 16 columns of the matrix instruction are those 8 rows (8
// columns) over the first half of K and over the second, so that two of the four 8 x 8 corners of its result are partial sums of the
// tile (the others are dropped: the matrix cores have nothing else to do).  Twice the workgroups, each with half the weights to
// fetch: a CU takes in about 45 KB/us here whatever the wavefronts and buffers, so that is what a long K waits for.
template <int MT, int NT, int KW, int D, int XR, int XM, bool EMIT, int H = 1>
__device__ __forceinline__ void gemm_ks_tile(const mm_args & a, const char * wb, const char * xb, char * db, const epi_args & epi, int64_t batch_off,
                                             int64_t d_nb1, int64_t m0, int64_t n0, half_t * x16) {
    constexpr int XE = XM == KS_X_F16 ? 2 : 4;
    constexpr int WL = 2 * MT, XL = XR * XE / 16;       // 1 KB loads per unit
    constexpr int UNIT_BYTES = (WL + XL) * 1024;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, q = lane >> 4;
    char * mine = smem + wave * (D * UNIT_BYTES);
    constexpr int MR = 16 * MT / H, NR = 16 * NT / H;
    const int64_t part = a.K / H;

    // load i covers lines 4 i .. + 3; this lane: line 4 i + lane / 16, slot lane % 16
    const char * wp[WL]; const char * xp[XL];
    auto row_of = [&](int i, int & chunk) __attribute__((always_inline)) { const int line = 4 * i + q; chunk = (lane & 7) ^ (line & 7); return 2 * line + ((lane >> 3) & 1); };
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        int c;
        const int r = row_of(i, c);
        const int64_t m = m0 + r % MR;
        wp[i] = wb + (m < a.M ? m : a.M - 1) * a.w_nb1 + c * 16 + r / MR * (part * 2);
    }
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        int c, r;
        if constexpr (XM == KS_X_F16) r = row_of(i, c);
        else { r = 4 * i + q; c = r16 ^ (r & 15); }
        const int64_t n = n0 + r % NR;
        xp[i] = xb + (n < a.N ? n : a.N - 1) * a.x_nb1 + c * 16 + r / NR * (part * XE);
    }
    auto load = [&](int64_t u, int buf) __attribute__((always_inline)) {
        char * to = mine + buf * UNIT_BYTES;
#pragma unroll
        for (int i = 0; i < WL; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(wp[i] + u * (KS_UNIT * 2)), (__attribute__((address_space(3))) void *)(to + i * 1024), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < XL; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(xp[i] + u * (KS_UNIT * XE)), (__attribute__((address_space(3))) void *)(to + (WL + i) * 1024), 16, 0, 0);
    };
    float4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (float4_t){ 0.f, 0.f, 0.f, 0.f };
    // fragment addresses inside a unit: f16 rows 16 i + r16 (line 8 i + r16 / 2), chunk 4 s + q
    const int frow = (r16 >> 1) * 256 + (r16 & 1) * 128, fsw = (r16 >> 1) & 7;
    auto mma = [&](int64_t u, int buf) __attribute__((always_inline)) {
        const char * ws = mine + buf * UNIT_BYTES, * xs = ws + WL * 1024;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int fo = frow + ((4 * s + q) ^ fsw) * 16;
            half8_t wv[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) wv[i] = *(const half8_t *)(ws + i * 2048 + fo);
            if constexpr (XM == KS_X_F16) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const half8_t xv = *(const half8_t *)(xs + j * 2048 + fo);
#pragma unroll
                    for (int i = 0; i < MT; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[i], xv, acc[i][j], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int r = XR == 8 ? r16 & 7 : r16;
                    const float4_t lo = *(const float4_t *)(xs + (16 * j + r) * 256 + ((8 * s + 2 * q) ^ r) * 16);
                    const float4_t hi = *(const float4_t *)(xs + (16 * j + r) * 256 + ((8 * s + 2 * q + 1) ^ r) * 16);
                    if constexpr (XM == KS_X_CVT) {
                        const half8_t xv = { (half_t) lo.x, (half_t) lo.y, (half_t) lo.z, (half_t) lo.w, (half_t) hi.x, (half_t) hi.y, (half_t) hi.z, (half_t) hi.w };
                        if (x16) {
                            const int rr = 16 * j + r16;
                            const int64_t n = n0 + rr % NR;
                            if (r16 < XR && n < a.N) *(half8_t *)(x16 + n * a.K + rr / NR * part + u * KS_UNIT + 32 * s + 8 * q) = xv;
                        }
#pragma unroll
                        for (int i = 0; i < MT; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[i], xv, acc[i][j], 0, 0, 0);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e)
#pragma unroll
                            for (int i = 0; i < MT; ++i)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32((float) wv[i][e], e < 4 ? lo[e & 3] : hi[e & 3], acc[i][j], 0, 0, 0);
                    }
                }
            }
        }
    };
    const int units = (int)(part / KS_UNIT), n_mine = units > wave ? (units - wave + KW - 1) / KW : 0;
#pragma unroll
    for (int t = 0; t < D - 1; ++t) if (t < n_mine) load(wave + t * KW, t);
    int t = 0, buf = 0;
    for (; t + D - 1 < n_mine; ++t) {
        load(wave + (int64_t)(t + D - 1) * KW, buf == 0 ? D - 1 : buf - 1);
        ks_wait_vmcnt<(D - 1) * (WL + XL)>();           // unit t is in LDS
        mma(wave + (int64_t) t * KW, buf);
        buf = buf + 1 == D ? 0 : buf + 1;
    }
    ks_wait_vmcnt<0>();
    for (; t < n_mine; ++t) { mma(wave + (int64_t) t * KW, buf); buf = buf + 1 == D ? 0 : buf + 1; }
    __syncthreads();                                    // (the partial tiles take the buffers' place)
    ks_finish<MT, NT, KW, EMIT, H>(acc, (float *) smem, a, db, epi, batch_off, d_nb1, m0, n0);
}

// k_gemm_k64: K = 64 (attention scores), more than a few tiles: the product is nothing beside the store of its result.  A wavefront
// keeps its 16 columns as fragments and walks `run` tiles of 64 rows, which its workgroup of four brings to LDS two tiles ahead;
// the results of a tile turn over in 4 KB of LDS of the wavefront's own and leave as 256-byte pieces of dst rows, behind which
// nobody waits: the wait for a tile counts the stores of the two tiles before it among what may still be on its way.
// 1500 x 1500, f32 columns, 12 heads: 25.5 us (a fill of the 108 MB: 18), with a workgroup of one wavefront to a 64 x 64 tile 30.5 — load,
// product, store, one behind the other, six to a CU; 20 heads 39.7; 44, 6 heads 15.5; 19.5, 227 columns of 20 heads 9.9; 13.2.
template <int XM>
__global__ void __launch_bounds__(256) k_gemm_k64(mm_args a, half_t * x16, int64_t x16_slice, int run) {
    constexpr int LD = 68;
    extern __shared__ __attribute__((aligned(16))) char smem[];     // [3][64 rows of 128 bytes], then [4][16 * LD] floats
    const mm_slice_ptrs z = mm_slice(a, blockIdx.z);
    char * db = a.d + z.d_off;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q = lane >> 4;
    const int64_t m0 = (int64_t) blockIdx.x * (64 * run), n0 = (int64_t) blockIdx.y * 64 + 16 * wave;
    const int tiles = (int) min((int64_t) run, (a.M - m0 + 63) / 64);

    // rows of a tile: the 1 KB loads 2 wave and 2 wave + 1 (layout of gemm_ks_tile)
    auto load = [&](int t, int buf) __attribute__((always_inline)) {
        t = min(t, tiles - 1);                              // (past the last tile: that one again, so that the count of what is on its way holds)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int line = 4 * (2 * wave + i) + q, row = 2 * line + ((lane >> 3) & 1);
            const int64_t m = min(m0 + 64 * t + row, a.M - 1);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(z.w + m * a.w_nb1 + ((lane & 7) ^ (line & 7)) * 16),
                                             (__attribute__((address_space(3))) void *)(smem + buf * 8192 + (2 * wave + i) * 1024), 16, 0, 0);
        }
    };
    half8_t xv[2];
    const int64_t n = n0 + r16;
    const char * xp = z.x + min(n, a.N - 1) * a.x_nb1;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if constexpr (XM == KS_X_F16) xv[s] = *(const half8_t *)(xp + (32 * s + 8 * q) * 2);
        else {
            const float4_t lo = *(const float4_t *)(xp + (32 * s + 8 * q) * 4), hi = *(const float4_t *)(xp + (32 * s + 8 * q) * 4 + 16);
            xv[s] = (half8_t){ (half_t) lo.x, (half_t) lo.y, (half_t) lo.z, (half_t) lo.w, (half_t) hi.x, (half_t) hi.y, (half_t) hi.z, (half_t) hi.w };
        }
    }
    if (XM == KS_X_CVT && x16 && blockIdx.x == 0 && n < a.N) {
#pragma unroll
        for (int s = 0; s < 2; ++s) *(half8_t *)(x16 + blockIdx.z * x16_slice + n * KS_UNIT + 32 * s + 8 * q) = xv[s];
    }
    ks_wait_vmcnt<0>();
    load(0, 0);
    load(1, 1);

    // four stores to a tile, no loads: what the counted waits assume (uniform)
    const bool counted = n0 + 16 <= a.N && !(a.e.flags & ~MI355X_EPI_SCALE);
    const float scale = a.e.flags & MI355X_EPI_SCALE ? a.e.scale : 1.0f;
    const int frow = (r16 >> 1) * 256 + (r16 & 1) * 128, fsw = (r16 >> 1) & 7;
    float * mine = (float *)(smem + 3 * 8192) + wave * (16 * LD);
    int buf = 0;
    for (int t = 0; t < tiles; ++t) {
        if (!counted)    ks_wait_vmcnt<0>();
        else if (t == 0) ks_wait_vmcnt<2>();
        else if (t == 1) ks_wait_vmcnt<2 + 4>();
        else             ks_wait_vmcnt<4 + 2 + 4>();
        __builtin_amdgcn_s_barrier();                       // everybody's pieces of tile t are in LDS; the buffer of tile t - 1 is free
        __builtin_amdgcn_sched_barrier(0);
        const char * ws = smem + buf * 8192;
        half8_t wv[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) wv[s][i] = *(const half8_t *)(ws + i * 2048 + frow + ((4 * s + q) ^ fsw) * 16);
        __builtin_amdgcn_sched_barrier(0);
        load(t + 2, buf == 0 ? 2 : buf - 1);
        __builtin_amdgcn_sched_barrier(0);
        float4_t acc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = (float4_t){ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[s][i], xv[s], acc[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) *(float4_t *)(mine + r16 * LD + 16 * i + 4 * q) = acc[i];
        const int64_t mt = m0 + 64 * t + 4 * r16;
        if (counted && m0 + 64 * t + 64 <= a.M) {
#pragma unroll
            for (int k = 0; k < 4; ++k) *(ks_f4 *)(db + (n0 + 4 * k + q) * a.d_nb1 + mt * 4) = *(const float4_t *)(mine + (4 * k + q) * LD + 4 * r16) * scale;
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float4_t v = *(const float4_t *)(mine + (4 * k + q) * LD + 4 * r16);
                if (n0 + 4 * k + q < a.N && mt < a.M) ks_store4<false>(v, mt, n0 + 4 * k + q, a, db, a.e, z.d_off, a.d_nb1);
            }
        }
        buf = buf == 2 ? 0 : buf + 1;
    }
    ks_wait_vmcnt<0>();                                     // (the surplus loads still write LDS)
}

template <int MT, int NT, int KW, int XM>
__device__ __forceinline__ void gemm_kd_tile(const mm_args & a, const char * wb, const char * xb, char * db, const epi_args & epi, int64_t batch_off,
                                             int64_t d_nb1, int64_t m0, int64_t n0) {
    constexpr int XE = XM == KS_X_F16 ? 2 : 4;          // bytes per src1 element
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float * red = (float *) smem;                       // [KW][16 NT][LD]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, q = lane >> 4;

    const char * wp[MT]; const char * xp[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) { const int64_t m = m0 + 16 * i + r16; wp[i] = wb + (m < a.M ? m : a.M - 1) * a.w_nb1 + q * 16; }
#pragma unroll
    for (int j = 0; j < NT; ++j) { const int64_t n = n0 + 16 * j + r16; xp[j] = xb + (n < a.N ? n : a.N - 1) * a.x_nb1 + q * 8 * XE; }

    struct frags { ks_h8 w[2][MT]; ks_h8 x[2][XM == KS_X_F16 ? NT : 1]; ks_f4 xf[2][XM == KS_X_F16 ? 1 : NT][2]; };
    float4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (float4_t){ 0.f, 0.f, 0.f, 0.f };

    auto load = [&](frags & f, int64_t u) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int64_t k = u * KS_UNIT + 32 * s;
#pragma unroll
            for (int i = 0; i < MT; ++i) f.w[s][i] = *(const ks_h8 *)(wp[i] + k * 2);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                if constexpr (XM == KS_X_F16) f.x[s][j] = *(const ks_h8 *)(xp[j] + k * 2);
                else { f.xf[s][j][0] = *(const ks_f4 *)(xp[j] + k * 4); f.xf[s][j][1] = *(const ks_f4 *)(xp[j] + k * 4 + 16); }
            }
        }
    };
    auto load_tail = [&](frags & f, int64_t u) __attribute__((always_inline)) {       // values past K are zero
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int64_t k = u * KS_UNIT + 32 * s;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool in = k + 8 * q + e < a.K;
                const int64_t at = in ? k + e : -(int64_t) 8 * q;                     // (k = 0 of the row, which exists)
#pragma unroll
                for (int i = 0; i < MT; ++i) { const half_t v = *(const half_t *)(wp[i] + at * 2); f.w[s][i][e] = in ? v : (half_t) 0.f; }
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    if constexpr (XM == KS_X_F16) { const half_t v = *(const half_t *)(xp[j] + at * 2); f.x[s][j][e] = in ? v : (half_t) 0.f; }
                    else { const float v = *(const float *)(xp[j] + at * 4); f.xf[s][j][e / 4][e % 4] = in ? v : 0.f; }
                }
            }
        }
    };
    auto mma = [&](const frags & f, int64_t u) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if constexpr (XM == KS_X_F32) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32((float) f.w[s][i][e], f.xf[s][j][e / 4][e % 4], acc[i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.w[s][i], f.x[s][j], acc[i][j], 0, 0, 0);
            }
        }
    };

    // Two units in flight.  Every load is unconditional (past the end it re-reads the last unit): with a load behind a
    // branch the compiler cannot count what is outstanding and waits for everything.
    const int64_t full = a.K / KS_UNIT;
    int64_t u = wave;
    if (u < full) {
        frags f0, f1;
        load(f0, u);
        while (true) {
            load(f1, u + KW < full ? u + KW : full - 1);
            mma(f0, u); u += KW; if (u >= full) break;
            load(f0, u + KW < full ? u + KW : full - 1);
            mma(f1, u); u += KW; if (u >= full) break;
        }
    }
    if (a.K % KS_UNIT != 0 && wave == (int)(full % KW)) {
        frags f;
        load_tail(f, full);
        mma(f, full);
    }

    ks_finish<MT, NT, KW, false>(acc, red, a, db, epi, batch_off, d_nb1, m0, n0);
}

// k_gemm_x32: f32 activations that stay f32 (the probabilities of plain attention against the transposed V of a head), many columns.
// v_mfma_f32_16x16x4_f32 multiplies them at a sixteenth of the bf16 rate, 22 us for 1500 x 1500 x 64 x 12 at its peak — as long as
// the 108 MB of activations take.  So a value goes to the bf16 matrix cores in three parts, its top eight significant bits, the
// next eight and the last eight (each a subtraction that loses nothing), a weight in two (f16 has eleven bits): six products of
// 32 steps where the f32 form takes eight of 4, 2.7 times the rate, every product exact and every sum f32 as before.
// A wavefront owns 16 columns and all 64 rows of the tile, so an activation is read and split once, straight from memory into
// the operand's lanes, three units of 64 ahead; the weights of a unit are split by the workgroup together and shared through LDS.
// A half unit's 24 matrix instructions take the splitting of the next half between them.  1500 x 1500 x 64, heads: 12 63 us -> 36
// (a K split over four wavefronts with f32 matrix instructions in front), 20 75 -> 45, 6 39 -> 25; 700 x 700 x 12 22 -> 14.
// (The activations through LDS, whole rows at a time, came out slower: 49 us.)
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t ks_u4 __attribute__((ext_vector_type(4)));
struct bf16_parts3 { ks_u4 hi, mid, lo; };
// the bf16 in the upper halves of two registers
__device__ __forceinline__ uint32_t pack_hi(float a, float b) { return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302); }
__device__ __forceinline__ float top_bf16(float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); }
__device__ __forceinline__ bf16_parts3 split3(const ks_f4 & x0, const ks_f4 & x1) {
    bf16_parts3 p;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = i < 2 ? x0[2 * i] : x1[2 * i - 4], b = i < 2 ? x0[2 * i + 1] : x1[2 * i - 3];
        const float ra = a - top_bf16(a), rb = b - top_bf16(b);
        p.hi[i] = pack_hi(a, b); p.mid[i] = pack_hi(ra, rb); p.lo[i] = pack_hi(ra - top_bf16(ra), rb - top_bf16(rb));
    }
    return p;
}

template <int NW>
__global__ void __launch_bounds__(64 * NW, 2) k_gemm_x32(mm_args a) {
    __shared__ __attribute__((aligned(16))) char w_lds[2][2][8192];       // [buffer][part][64 rows of 128 bytes, chunks swizzled as in gemm_ks_tile]
    const mm_slice_ptrs z = mm_slice(a, blockIdx.z);
    const int64_t m0 = (int64_t) blockIdx.x * 64, n0 = (int64_t) blockIdx.y * (16 * NW);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, q = lane >> 4;
    const int units = (int)(a.K / KS_UNIT), tail = (int)(a.K % KS_UNIT);      // whole ones; values behind them
    const int64_t n = n0 + 16 * wave + r16;
    const char * xp = z.x + (n < a.N ? n : a.N - 1) * a.x_nb1 + q * 32;
    // this thread's weights of a unit: WC chunks of 8 values, of row wr[i] chunk wc
    constexpr int WC = (512 + 64 * NW - 1) / (64 * NW);    // (512 chunks of 8 values in a unit)
    int wr[WC], wc[WC]; const char * wp[WC]; bool w_ok[WC];
#pragma unroll
    for (int i = 0; i < WC; ++i) {
        const int c = i * 64 * NW + tid;
        w_ok[i] = 512 % (64 * NW) == 0 || c < 512;
        wr[i] = (c >> 3) & 63; wc[i] = c & 7;
        wp[i] = z.w + (m0 + wr[i] < a.M ? m0 + wr[i] : a.M - 1) * a.w_nb1 + wc[i] * 16;
    }

    struct xunit { ks_f4 v[2][2]; };
    struct wunit { ks_h8 v[WC]; };
    // (units past the end re-read the last one: no load behind a branch, which would be waited for with every other)
    auto load_x = [&](xunit & x, int u) __attribute__((always_inline)) {
        const int64_t k = (int64_t)(u < units ? u : units - 1) * (KS_UNIT * 4);
#pragma unroll
        for (int s = 0; s < 2; ++s) { x.v[s][0] = *(const ks_f4 *)(xp + k + 128 * s); x.v[s][1] = *(const ks_f4 *)(xp + k + 128 * s + 16); }
    };
    auto load_w = [&](wunit & w, int u) __attribute__((always_inline)) {
        const int64_t k = (int64_t)(u < units ? u : units - 1) * (KS_UNIT * 2);
#pragma unroll
        for (int i = 0; i < WC; ++i) w.v[i] = *(const ks_h8 *)(wp[i] + k);
    };
    auto store_w = [&](const wunit & w, int buf, int i) __attribute__((always_inline)) {
        ks_u4 hi, lo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = (float) w.v[i][2 * e], y = (float) w.v[i][2 * e + 1];
            hi[e] = pack_hi(x, y); lo[e] = pack_hi(x - top_bf16(x), y - top_bf16(y));
        }
        char * to = &w_lds[buf][0][0] + (wr[i] >> 1) * 256 + (wr[i] & 1) * 128 + (wc[i] ^ ((wr[i] >> 1) & 7)) * 16;
        if (w_ok[i]) { *(ks_u4 *) to = hi; *(ks_u4 *)(to + 8192) = lo; }
    };
    float4_t acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = (float4_t){ 0.f, 0.f, 0.f, 0.f };
    const int frow = (r16 >> 1) * 256 + (r16 & 1) * 128, fsw = (r16 >> 1) & 7;
    struct wfrag { bf16x8_t h[4], l[4]; };
    auto read_w = [&](wfrag & w, int buf, int s) __attribute__((always_inline)) {
        const char * at = &w_lds[buf][0][0] + frow + ((4 * s + q) ^ fsw) * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) { w.h[i] = *(const bf16x8_t *)(at + i * 2048); w.l[i] = *(const bf16x8_t *)(at + i * 2048 + 8192); }
    };
    auto mma = [&](const wfrag & w, const bf16_parts3 & p) __attribute__((always_inline)) {
        const bf16x8_t xh = __builtin_bit_cast(bf16x8_t, p.hi), xm = __builtin_bit_cast(bf16x8_t, p.mid), xl = __builtin_bit_cast(bf16x8_t, p.lo);
        // (the small products first)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.l[i], xl, acc[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.h[i], xl, acc[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.l[i], xm, acc[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.h[i], xm, acc[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.l[i], xh, acc[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.h[i], xh, acc[i], 0, 0, 0);
    };
    // issue order of a half unit: a matrix instruction, then what fits into its time of the splitting for the next half
    auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 24; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                      // 1 matrix instruction
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);                      // 4 vector instructions
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    xunit x[4]; wunit w[2];
    bf16_parts3 p0, p1;
    if (units > 0) {                                       // uniform
        load_w(w[0], 0); load_x(x[0], 0);
        load_w(w[1], 1); load_x(x[1], 1);
#pragma unroll
        for (int i = 0; i < WC; ++i) store_w(w[0], 0, i);
        load_w(w[0], 2); load_x(x[2], 2);
        p0 = split3(x[0].v[0][0], x[0].v[0][1]);
        __syncthreads();
        // unit u: x[u % 4], its first half split already; w[(u + 1) % 2] holds the weights of unit u + 1
        auto step = [&](int u, xunit & cur, const xunit & nxt, xunit & far, wunit & wn) __attribute__((always_inline)) {
            wfrag f0, f1;
            read_w(f0, u & 1, 0);
            load_x(far, u + 3);
            __builtin_amdgcn_sched_barrier(0);
            read_w(f1, u & 1, 1);
            p1 = split3(cur.v[1][0], cur.v[1][1]);
            mma(f0, p0);
#pragma unroll
            for (int i = 0; i < WC / 2; ++i) store_w(wn, (u + 1) & 1, i);
            interleave();
            p0 = split3(nxt.v[0][0], nxt.v[0][1]);
            mma(f1, p1);
#pragma unroll
            for (int i = WC / 2; i < WC; ++i) store_w(wn, (u + 1) & 1, i);
            interleave();
#pragma unroll
            for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(p0.hi[i]), "+v"(p0.mid[i]), "+v"(p0.lo[i]));       // (split here, not where it is used)
            load_w(wn, u + 3);
            __syncthreads();
        };
        for (int u = 0;;) {
            step(u, x[0], x[1], x[3], w[1]); if (++u >= units) break;
            step(u, x[1], x[2], x[0], w[0]); if (++u >= units) break;
            step(u, x[2], x[3], x[1], w[1]); if (++u >= units) break;
            step(u, x[3], x[0], x[2], w[0]); if (++u >= units) break;
        }
    }
    if (tail != 0) {                                       // the unit that K ends in: value by value, zeros behind the end
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int k = 32 * s + 8 * q + e;
                const float v = *(const float *)(xp - q * 32 + (k < tail ? (int64_t) units * KS_UNIT + k : 0) * 4);
                x[0].v[s][e / 4][e % 4] = k < tail ? v : 0.0f;
            }
#pragma unroll
        for (int i = 0; i < WC; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int k = 8 * wc[i] + e;
                const half_t v = *(const half_t *)(wp[i] - wc[i] * 16 + (k < tail ? (int64_t) units * KS_UNIT + k : 0) * 2);
                w[0].v[i][e] = k < tail ? v : (half_t) 0.0f;
            }
#pragma unroll
        for (int i = 0; i < WC; ++i) store_w(w[0], 0, i);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            wfrag f;
            read_w(f, 0, s);
            mma(f, split3(x[0].v[s][0], x[0].v[s][1]));
        }
    }

    if (n >= a.N) return;
    char * db = a.d + z.d_off;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t m = m0 + 16 * i + 4 * q;
        if (a.e.flags == 0 && m + 3 < a.M) { *(ks_f4 *)(db + n * a.d_nb1 + m * 4) = (ks_f4){ acc[i][0], acc[i][1], acc[i][2], acc[i][3] }; continue; }
        for (int e = 0; e < 4 && m + e < a.M; ++e) {
            const float v = apply_epilogue(acc[i][e], a.e, m + e, n, z.d_off + n * a.d_nb1 + (m + e) * 4);
            if (a.e.flags & MI355X_EPI_OUT_F16) *(half_t *)(db + n * a.d_nb1 + (m + e) * 2) = (half_t) v;
            else                                *(float  *)(db + n * a.d_nb1 + (m + e) * 4) = v;
        }
    }
}

// grids: m tiles x n tiles x batch
#define KS_SLICES const mm_slice_ptrs z = mm_slice(a, blockIdx.z); const char * wb = z.w, * xb = z.x; const int64_t d_off = z.d_off; \
    const int64_t m0 = (int64_t) blockIdx.x * (16 * MT / H), n0 = (int64_t) blockIdx.y * (16 * NT / H);

template <int MT, int NT, int KW, int D, int XR, int XM, bool EMIT, int H>
__global__ void __launch_bounds__(64 * KW) k_gemm_ks(mm_args a, half_t * x16, int64_t x16_slice) {
    KS_SLICES
    gemm_ks_tile<MT, NT, KW, D, XR, XM, EMIT, H>(a, wb, xb, a.d + d_off, a.e, d_off, a.d_nb1, m0, n0, x16 && blockIdx.x == 0 ? x16 + blockIdx.z * x16_slice : nullptr);
}
// several products over the same activations: blockIdx.z picks the weights, the destination and the epilogue
struct ks_group { mm_group_entry e[KS_GROUP_MAX]; };
template <int MT, int NT, int KW, int D, int XR, int XM, int H>
__global__ void __launch_bounds__(64 * KW) k_gemm_ks_group(mm_args a, ks_group grp, half_t * x16) {
    const mm_group_entry & ge = grp.e[blockIdx.z];
    epi_args e;
    e.flags = ge.flags; e.scale = ge.scale; e.bias = ge.bias; e.residual = ge.residual; e.gelu = a.e.gelu; e.image = nullptr;
    gemm_ks_tile<MT, NT, KW, D, XR, XM, false, H>(a, ge.w, a.x, ge.d, e, 0, ge.d_nb1, (int64_t) blockIdx.x * (16 * MT / H), (int64_t) blockIdx.y * (16 * NT / H),
                                               blockIdx.x == 0 && blockIdx.z == 0 ? x16 : nullptr);
}
template <int MT, int NT, int KW, int XM>
__global__ void __launch_bounds__(64 * KW) k_gemm_kd(mm_args a) {
    constexpr int H = 1;
    KS_SLICES
    gemm_kd_tile<MT, NT, KW, XM>(a, wb, xb, a.d + d_off, a.e, d_off, a.d_nb1, m0, n0);
}

template <int MT, int NT, int H = 1>
static int ks_grid(const mm_args & a, dim3 & grid) {
    const int64_t tm = (a.M + 16 * MT / H - 1) / (16 * MT / H), tn = (a.N + 16 * NT / H - 1) / (16 * NT / H), nb = a.ne12 * a.ne13;
    if (tm > 0x7fffffff || tn > 65535 || nb > 65535) return MI355X_ERR_UNSUPPORTED;
    grid = dim3((unsigned) tm, (unsigned) tn, (unsigned) nb);
    return MI355X_OK;
}
// more than the default 64 KB of LDS have to be asked for, once per kernel and device
static int ks_configure(const void * fn, size_t lds, std::atomic<bool> * configured) {
    if (lds <= 64 * 1024) return MI355X_OK;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return MI355X_ERR_HIP;
    if (configured[dev].load(std::memory_order_acquire)) return MI355X_OK;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds) != hipSuccess) return MI355X_ERR_HIP;
    configured[dev].store(true, std::memory_order_release);
    return MI355X_OK;
}

template <int MT, int NT, int KW, int D, int XR, int XM, bool EMIT, int H = 1>
static int launch_ks_t(const mm_args & a, half_t * x16, int64_t slice, hipStream_t st) {
    constexpr size_t ring = (size_t) KW * D * (2 * MT + XR * (XM == KS_X_F16 ? 2 : 4) / 16) * 1024, red = ks_red_bytes<MT, NT, KW>(), lds = ring > red ? ring : red;
    static std::atomic<bool> configured[64];
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    dim3 grid;
    if (int rc = ks_grid<MT, NT, H>(a, grid)) return rc;
    if (int rc = ks_configure((const void *) k_gemm_ks<MT, NT, KW, D, XR, XM, EMIT, H>, lds, configured)) return rc;
    k_gemm_ks<MT, NT, KW, D, XR, XM, EMIT, H><<<grid, 64 * KW, lds, st>>>(a, x16, slice);
    return launch_status();
}
template <int MT, int NT, int KW, int XM>
static int launch_kd_t(const mm_args & a, hipStream_t st) {
    constexpr size_t lds = ks_red_bytes<MT, NT, KW>();
    static std::atomic<bool> configured[64];
    dim3 grid;
    if (int rc = ks_grid<MT, NT>(a, grid)) return rc;
    if (int rc = ks_configure((const void *) k_gemm_kd<MT, NT, KW, XM>, lds, configured)) return rc;
    k_gemm_kd<MT, NT, KW, XM><<<grid, 64 * KW, lds, st>>>(a);
    return launch_status();
}
template <int XM>
static int launch_k64(const mm_args & a, half_t * x16, int64_t slice, hipStream_t st) {
    const int64_t t = (a.M + 63) / 64, tn = (a.N + 63) / 64, nb = a.ne12 * a.ne13;
    const int run = (t + 5) / 6 * tn * nb >= 512 ? 6 : 4;           // (700 x 700, 12 heads: 11.4 us with 6, 9.9 with 4)
    const int64_t tm = (t + run - 1) / run;
    if (tm > 0x7fffffff || tn > 65535 || nb > 65535) return MI355X_ERR_UNSUPPORTED;
    k_gemm_k64<XM><<<dim3((unsigned) tm, (unsigned) tn, (unsigned) nb), 256, 3 * 8192 + 4 * 16 * 68 * 4, st>>>(a, x16, slice, run);
    return launch_status();
}
template <int XM, bool EMIT>
static int launch_ks_x(const mm_args & a, const ks_shape & s, half_t * x16, int64_t slice, hipStream_t st) {
    const bool few = a.N <= 8;
#define KS_CASE(MT, NT, KW, D) if (s.h == 1 && s.mt == MT && s.nt == NT && s.kw == KW && s.d == D) { if constexpr (!EMIT || MT % 2 == 0) { \
        if constexpr (NT == 1) if (few) return launch_ks_t<MT, NT, KW, D, 8, XM, EMIT>(a, x16, slice, st); \
        return launch_ks_t<MT, NT, KW, D, 16 * NT, XM, EMIT>(a, x16, slice, st); } }
#define KS_HALVES(KW, D) if (s.h == 2 && s.kw == KW && s.d == D) { if constexpr (!EMIT) return launch_ks_t<1, 1, KW, D, 16, XM, EMIT, 2>(a, x16, slice, st); }
    KS_HALVES(4, 2) KS_HALVES(8, 2)
#undef KS_HALVES
    KS_CASE(1, 1, 1, 1) KS_CASE(1, 1, 4, 2) KS_CASE(1, 1, 8, 2) KS_CASE(2, 1, 4, 2)
    if constexpr (XM != KS_X_F32) {
        KS_CASE(2, 2, 1, 1)
        if constexpr (!EMIT) if (s.kw == 1 && s.mt == 4) return launch_k64<XM>(a, x16, slice, st);
    }
    if constexpr (XM == KS_X_F16) { KS_CASE(2, 2, 4, 2) KS_CASE(4, 4, 4, 2) }
#undef KS_CASE
    return MI355X_ERR_UNSUPPORTED;
}

// Tile and split by size (MI355X, weights from HBM, us per launch; "128-wide" is what the tiled kernels of mul_mat.hip take):
//   up to 16 columns: 16 x 16 tiles, 8 wavefronts on their K range (1280 x 1280, 5 columns: 4.1, with 4 4.5, 64 x 64 tiles 10.3;
//     1280 x 5120: 9.4; 11.1; 26.3), above 4096 rows 32 rows to a tile and 4 wavefronts (51866 x 1280: 26.3; 16 rows 28.0; 40.4);
//   up to 8 columns and 2048 rows, where 16-row tiles leave half the CUs idle: 8-row tiles (H = 2), 8 wavefronts from K = 1024 on
//     (1280 x 5120: 7.8; 1024 x 4096: 6.7, 16-row tiles 7.9; 1280 x 1280: 3.9; 512 x 512: 2.9, 16-row tiles 3.1; at 3072 x 768 they
//     lose, 6.1 to 4.2);
//   one round of 64 x 64 tiles, at least half of one (M = 512, K = 2048, N = 1500: 12.9; 128-wide 14.3; M = 1280, K = 1280,
//     N = 700: 10.2; 11.3), else 32 x 32 (1280 x 5120, 227 columns: 17.8; 34.9; 384 x 384, 487 columns: 3.9; 7.3), and 16 x 16 where
//     that is under half a round as well (768 x 768, 27 columns: 3.7; 4.4; 6.8);
//   more than a round of 64 x 64 tiles: the 128-wide tiles, which move half the bytes per product (M = 768, N = 1500: 8.9;
//     10.7 here), except with up to 32 columns, where they are mostly padding (51865 x 768, 27 columns: 21.7; 23.9).
// K = 64 (attention scores) is one unit: no split, one wavefront to a tile; from 512 64 x 64 tiles on k_gemm_k64, for the store of the result.
static bool ks_tiles(int64_t M, int64_t N, int64_t K, int64_t nb, bool emit, ks_shape & s) {
    const int64_t t44 = (M + 63) / 64 * ((N + 63) / 64) * nb, t22 = (M + 31) / 32 * ((N + 31) / 32) * nb;
    s.kw = 4; s.d = 2; s.h = 1;
    if (K == KS_UNIT) {
        s.kw = 1; s.d = 1;
        s.mt = s.nt = N <= 16 || t22 < 512 ? 1 : t44 < 512 ? 2 : 4;
        return !emit;
    }
    if (N <= 16) {
        s.nt = 1; s.mt = emit || M > 4096 ? 2 : 1;
        if (s.mt == 1 && N <= 8 && M <= 2048 && nb == 1 && K % (2 * KS_UNIT) == 0) { s.h = 2; s.kw = K >= 1024 ? 8 : 4; }
        else if (s.mt == 1) s.kw = 8;
        return true;
    }
    if (t44 > 256) { s.mt = s.nt = 2; return N <= 32; }
    s.mt = s.nt = t44 > 128 ? 4 : t22 > 128 ? 2 : 1;
    if (emit && s.mt == 1) s.mt = 2;
    return true;
}
bool ks_pick(int64_t M, int64_t N, int64_t K, int64_t nb, bool emit, ks_shape & s) {
    return K > 0 && K % KS_UNIT == 0 && ks_tiles(M, N, K, nb, emit, s);
}
// A group of up to 8 columns is a product with the rows of all of them.  One of more columns goes the way of its single products,
// on tiles chosen for all of them together; the K split, and with it the order of the sums, is the same for every tile size.  A
// group that fills the device with 128-wide tiles goes there.
bool ks_pick_group(int64_t M, int64_t N, int64_t K, int count, ks_shape & s) {
    ks_shape one;
    if (count > KS_GROUP_MAX || !ks_pick(M, N, K, 1, false, one)) return false;
    if (N <= 8) return ks_pick(M * count, N, K, 1, false, s);
    return ks_pick(M, N, K, count, false, s) && s.kw == one.kw;
}
bool ks_converts(const ks_shape & s) { return s.nt == 1 || s.kw == 1; }

int launch_gemm_ks(const mm_args & a, const ks_shape & s, int xm, half_t * x16, int64_t x16_slice, hipStream_t st) {
    const bool emit = a.e.flags & MI355X_EPI_EMIT_F16;
    switch (xm) {
        case KS_X_F16: return emit ? launch_ks_x<KS_X_F16, true>(a, s, x16, x16_slice, st) : launch_ks_x<KS_X_F16, false>(a, s, x16, x16_slice, st);
        case KS_X_CVT: return emit ? MI355X_ERR_UNSUPPORTED : launch_ks_x<KS_X_CVT, false>(a, s, x16, x16_slice, st);
        default:       return emit ? MI355X_ERR_UNSUPPORTED : launch_ks_x<KS_X_F32, false>(a, s, x16, x16_slice, st);
    }
}

template <int MT, int NT, int KW, int D, int XR, int XM, int H>
static int launch_ks_group_t(const mm_args & a, const ks_group & grp, int count, half_t * x16, hipStream_t st) {
    constexpr size_t ring = (size_t) KW * D * (2 * MT + XR * (XM == KS_X_F16 ? 2 : 4) / 16) * 1024, red = ks_red_bytes<MT, NT, KW>(), lds = ring > red ? ring : red;
    static std::atomic<bool> configured[64];
    dim3 grid;
    if (int rc = ks_grid<MT, NT, H>(a, grid)) return rc;
    grid.z = (unsigned) count;
    if (int rc = ks_configure((const void *) k_gemm_ks_group<MT, NT, KW, D, XR, XM, H>, lds, configured)) return rc;
    k_gemm_ks_group<MT, NT, KW, D, XR, XM, H><<<grid, 64 * KW, lds, st>>>(a, grp, x16);
    return launch_status();
}
template <int MT, int NT, int KW, int D, int XR, int H = 1>
static int launch_ks_group_x(const mm_args & a, const ks_group & grp, int count, half_t * x16, hipStream_t st) {
    if constexpr (NT == 1) if (x16) return launch_ks_group_t<MT, NT, KW, D, XR, KS_X_CVT, H>(a, grp, count, x16, st);
    return x16 ? MI355X_ERR_UNSUPPORTED : launch_ks_group_t<MT, NT, KW, D, XR, KS_X_F16, H>(a, grp, count, x16, st);
}
int launch_gemm_ks_group(const mm_args & a, const mm_group & all, int count, const ks_shape & s, half_t * x16, hipStream_t st) {
    ks_group grp;
    for (int i = 0; i < count; ++i) grp.e[i] = all.e[i];
    if (s.h == 2) return s.kw == 8 ? launch_ks_group_x<1, 1, 8, 2, 16, 2>(a, grp, count, x16, st) : launch_ks_group_x<1, 1, 4, 2, 16, 2>(a, grp, count, x16, st);
#define KS_CASE(MT, NT, KW, D) if (s.mt == MT && s.nt == NT && s.kw == KW && s.d == D) { \
        if constexpr (NT == 1) if (a.N <= 8) return launch_ks_group_x<MT, NT, KW, D, 8>(a, grp, count, x16, st); \
        return launch_ks_group_x<MT, NT, KW, D, 16 * NT>(a, grp, count, x16, st); }
    KS_CASE(1, 1, 4, 2) KS_CASE(1, 1, 8, 2) KS_CASE(2, 1, 4, 2) KS_CASE(2, 2, 4, 2) KS_CASE(4, 4, 4, 2)
#undef KS_CASE
    return MI355X_ERR_UNSUPPORTED;
}

// The direct kernel, by size: a few columns on 16 x 16 tiles with as many wavefronts as the K range has units, up to 8; more
// on 64 x 32 (64 rows are all there are of the transposed V of a head: src1 is then read once), or k_gemm_x32 where src1 stays f32.
int launch_gemm_kd(const mm_args & a, int xm, hipStream_t st) {
    const bool few = a.N <= 16;
    const int kw = a.K <= KS_UNIT ? 1 : a.K < 8 * KS_UNIT ? 4 : 8;
    if (xm == KS_X_F16) {
        if (!few) return launch_kd_t<4, 2, 4, KS_X_F16>(a, st);
        return kw == 1 ? launch_kd_t<1, 1, 1, KS_X_F16>(a, st) : kw == 4 ? launch_kd_t<1, 1, 4, KS_X_F16>(a, st) : launch_kd_t<1, 1, 8, KS_X_F16>(a, st);
    }
    if (!few) {
        // as many wavefronts to the workgroup, 4, 5 or 6, as deal the 16-column pieces out to the CUs most evenly
        const int64_t tm = (a.M + 63) / 64, nb = a.ne12 * a.ne13;
        int nw = 4; int64_t best = INT64_MAX;
        for (int i : { 4, 5, 6 }) {
            const int64_t cost = (tm * ((a.N + 16 * i - 1) / (16 * i)) * nb + 255) / 256 * i;
            if (cost < best) { best = cost; nw = i; }
        }
        const int64_t tn = (a.N + 16 * nw - 1) / (16 * nw);
        if (tm > 0x7fffffff || tn > 65535 || nb > 65535) return MI355X_ERR_UNSUPPORTED;
        const dim3 grid((unsigned) tm, (unsigned) tn, (unsigned) nb);
        switch (nw) {
            case 4:  k_gemm_x32<4><<<grid, 256, 0, st>>>(a); break;
            case 5:  k_gemm_x32<5><<<grid, 320, 0, st>>>(a); break;
            default: k_gemm_x32<6><<<grid, 384, 0, st>>>(a); break;
        }
        return launch_status();
    }
    return kw == 1 ? launch_kd_t<1, 1, 1, KS_X_F32>(a, st) : kw == 4 ? launch_kd_t<1, 1, 4, KS_X_F32>(a, st) : launch_kd_t<1, 1, 8, KS_X_F32>(a, st);
}
