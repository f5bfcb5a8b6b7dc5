// factor.h -- the kernels of factor.hip, a translation unit of its own.
#pragma once
#include "sunhip_kernels.h"

#define FPB 16      // panel width
#define FTW 4       // 16-row tiles per wave: NW waves hold 64 NW rows
#define FLMAX 512   // largest N of the square forms (eight waves)

// scalar slots that the QR of a tall matrix fills: log|det R| and the count of negative diagonal entries
enum { SC_RLOG = 30, SC_RNEG = 31 };

// nc: 0 for the chain's N x N matrix, else its columns
template <int NW, int FT>
__global__ void k_qr_step(const DChain *chains, int sel, int k, int out_pt, int nc);
template <int NW, int FT>
__global__ void k_formq_cb(const DChain *chains, int nch, int ncb, int sel, int out_pt, int nc);
template <int NW>
__global__ void k_lu_step(const DChain *chains, int k, int zslot, int fresh);
