// Host launchers of the wave-row kernels (tcq_blocks.hip), called by the row entry points of tcq_walsh.hip after their
// argument checks. Each returns false, launching nothing, for rows it does not take. lds: the LDS engine would run these rows in whole
// 16-byte vectors (element by element it is far slower than the wave rows at any width).
#pragma once
#include "tcq_device.h"

bool blocks_rht(const void* x, int x_dtype, int ldx, const i8* su, void* y, int y_dtype, int ldy, int M, int K, hipStream_t st);
bool blocks_pre(const void* x, int x_dtype, const i8* su, const u16* cs, i8* q, int* q4, int ldq, float* scale, int M, int K, bool lds,
                hipStream_t st);
bool blocks_post(const tcq_post_seg* segs, int nseg, int acc_dtype, const float* s, const u16* gelu_lut, int y_dtype, int M,
                 bool lds, hipStream_t st);
bool blocks_mid1(const void* acc, int acc_dtype, int lda, const float* s, const float* rs, const i8* sv, const float* bias,
                 const u16* lut, const i8* su, i8* q, int* q4, int ldq, float* scale, int M, int N, bool lds, hipStream_t st);
