// Argument blocks of the MUL_MAT kernels (shared by mul_mat.hip and the harness-only instances of its kernels).
#pragma once

#include "common.h"

typedef uint32_t __attribute__((aligned(2))) u32a2;
struct __attribute__((packed, aligned(2))) u128a2 { uint32_t x, y, z, w; };
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int      v4i_t __attribute__((ext_vector_type(4)));

struct epi_args {
    int          flags;
    float        scale;
    const float *bias;
    const char * residual;   // same strides as dst, f32
    const uint16_t * gelu;   // GELU table (device), set when MI355X_EPI_GELU is
    half_t * image;          // MI355X_EPI_EMIT_F16: where the Q8_0-rounded f16 image of dst goes ([N][M] dense)
};

struct mm_args {
    const char * w; const char * x; char * d;
    int64_t M, N, K;
    int64_t w_nb1, w_nb2, w_nb3;
    int64_t x_nb1, x_nb2, x_nb3;
    int64_t d_nb1, d_nb2, d_nb3;
    int64_t ne12, ne13, r2, r3;      // batch dims of src1/dst and broadcast ratios of src0
    epi_args e;
};

// one product of a grouped launch
#define MM_GROUP_MAX 64
struct mm_group_entry { const char * w; char * d; const float * bias; const char * residual; int64_t d_nb1; int flags; float scale; };
struct mm_group { mm_group_entry e[MM_GROUP_MAX]; };

#ifdef __HIPCC__
// the operands of batch slice z (z = b2 + ne12 b3)
struct mm_slice_ptrs { const char * w; const char * x; int64_t d_off; };
__device__ __forceinline__ mm_slice_ptrs mm_slice(const mm_args & a, uint32_t z) {
    const uint32_t b3 = a.ne13 == 1 ? 0 : div_count(z, a.ne12), b2 = z - b3 * (uint32_t) a.ne12;
    return { a.w + div_count(b2, a.r2) * a.w_nb2 + div_count(b3, a.r3) * a.w_nb3, a.x + b2 * a.x_nb2 + b3 * a.x_nb3, b2 * a.d_nb2 + b3 * a.d_nb3 };
}
// four bits -> bit 4 of four bytes
__device__ __forceinline__ uint32_t spread4_to_bit4(uint32_t nib) {
    return ((nib * 0x00204081u) & 0x01010101u) << 4;
}
// epilogue of one value
__device__ __forceinline__ float apply_epilogue(float v, const epi_args & e, int64_t m, int64_t n, int64_t res_off) {
    if (e.flags & MI355X_EPI_BIAS)     v += e.bias[m];
    if (e.flags & MI355X_EPI_BIAS_COL) v += e.bias[n];
    if (e.flags & MI355X_EPI_GELU)     v  = gelu_f32(v, e.gelu);
    if (e.flags & MI355X_EPI_SCALE)    v *= e.scale;
    if (e.flags & MI355X_EPI_RESIDUAL) v += *(const float *)(e.residual + res_off);
    return v;
}
#endif
