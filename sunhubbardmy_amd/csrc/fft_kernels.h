// fft_kernels.h -- the kernels of fft_kernels.hip, a translation unit of its own.
#pragma once
#include "sunhip_kernels.h"

// padded length of one vector in LDS
__host__ __device__ __forceinline__ int fft_ld(int n, int n0)
{
    const int ld = n + n / n0;
    return ld | 1;
}
extern "C" __global__ void k_fft_cols(const DChain *chains, int msel, int pt, int ksel, int prog, int vsel, int nt0, int nt1, int ntstep, int fcb);
extern "C" __global__ void k_fft_rows(const DChain *chains, int msel, int pt, int ksel, int prog, int vsel, int nt, int fcb);
