// The split-K product over f16 weights (gemm_ks.hip) as mul_mat.hip launches it.
#pragma once

#include "mul_mat_args.h"

enum { KS_X_F16 = 0,        // src1 is f16 rows (or their f16 image in the workspace)
       KS_X_CVT = 1,        // src1 is f32, rounded to f16 on its way into the fragments; the first workgroup column also leaves
                            // the f16 rows in the workspace (what MI355X_MM_WS_READY of a later call refers to)
       KS_X_F32 = 2 };      // src1 is f32 and stays f32: v_mfma_f32_16x16x4_f32 on the widened weights (exact products)

struct ks_shape { int mt, nt, kw, d, h; };      // tile of 16 mt x 16 nt results (h = 2: of 8 x 8), kw wavefronts that share its K range, d buffers each
#define KS_GROUP_MAX 8

// false: the tiled kernels of mul_mat.hip are the better ones for this size (or K is no multiple of 64)
bool ks_pick(int64_t M, int64_t N, int64_t K, int64_t nb, bool emit, ks_shape & s);
bool ks_pick_group(int64_t M, int64_t N, int64_t K, int count, ks_shape & s);
bool ks_converts(const ks_shape & s);           // the shape has a KS_X_CVT form
// rows of src0 and src1 16-byte aligned; a.x: src1 (KS_X_CVT, KS_X_F32) or its f16 rows
int launch_gemm_ks(const mm_args & a, const ks_shape & s, int xm, half_t * x16, int64_t x16_slice, hipStream_t st);
// x16: a.x is f32 (KS_X_CVT) and its f16 rows go there; NULL: a.x is f16 rows
int launch_gemm_ks_group(const mm_args & a, const mm_group & all, int count, const ks_shape & s, half_t * x16, hipStream_t st);
// any alignment, any K
int launch_gemm_kd(const mm_args & a, int xm, hipStream_t st);
