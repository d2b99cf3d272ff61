/* ckq_gemm_f32act.hpp - entry of ckq_gemm_f32act.hip */
#pragma once
#include "ckq_formats.hpp"
int launch_gemm_f32act(int fmt, const float *A, const void *B, const float *bias, float *C, int M, int N, int K, long ldc, hipStream_t s);
