// What mul_mat.hip and gemv.hip share on the host: which kernel family a product runs on, and the few-column launches.
#pragma once

#include "mul_mat_args.h"

enum { MM_GENERIC = 0, MM_GEMV = 1, MM_GEMM = 2 };
int mm_path(const mi355x_tensor * src0, const mi355x_tensor * src1);

static inline size_t round256(size_t n) { return (n + 255) / 256 * 256; }
static inline bool aligned16(const mi355x_tensor * t) {
    return (uintptr_t) t->data % 16 == 0 && t->nb[1] % 16 == 0 && t->nb[2] % 16 == 0 && t->nb[3] % 16 == 0;
}

// bytes of the quantized activations that the register kernels read (0: the shape runs with in-kernel quantization)
size_t gemv_ws_bytes(const mi355x_tensor * src0, const mi355x_tensor * src1);
int launch_quantize_x_q8(const char * x, int64_t x_nb1, int64_t K, int64_t N, char * ws, hipStream_t st);
int launch_gemv_ws(int type, const mm_args & a, hipStream_t st);       // a.x: the activations as launch_quantize_x_q8 leaves them
int launch_gemv_lds(int type, const mm_args & a, hipStream_t st);      // a.x: f32 activations, quantized by every workgroup for itself
int mul_mat_group_gemv(const mi355x_mul_mat_item * items, int count, const mi355x_tensor * src1, int flags, void * workspace, size_t workspace_size, void * stream);
