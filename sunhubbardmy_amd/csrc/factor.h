// factor.h -- the kernels of factor.hip, a translation unit of its own.
#pragma once
#include "sunhip_kernels.h"

#define FPB 16      // panel width
#define FTW 4       // 16-row tiles per wave: NW waves hold 64 NW rows
#define FLMAX 512   // largest N (eight waves)

template <int NW>
__global__ void k_qr_step(const DChain *chains, int sel, int k, int out_pt);
template <int NW>
__global__ void k_formq_cb(const DChain *chains, int nch, int ncb, int sel, int out_pt);
template <int NW>
__global__ void k_lu_step(const DChain *chains, int k);
