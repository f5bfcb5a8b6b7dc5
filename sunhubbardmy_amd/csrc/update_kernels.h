// update_kernels.h -- the kernels of update_kernels.hip, a translation unit of its own.
#pragma once
#include "exchange.h"

template <int NT, bool WHOLE, int NF>
__global__ void k_upd_sites(const DChain *chains, int nt, int slice_in_pass, int s0);
template <int NT>
__global__ void k_upd_bonds(const DChain *chains, int nt, int nf, int slice, int p, int ib0, int per);
extern "C" __global__ void k_upd_panel(const DChain *chains, int s0);
extern "C" __global__ void k_upd_flush(const DChain *chains, int nch, int nt, int s0);
extern "C" __global__ void k_upd_panel_small(const DChain *chains, int nch, int grp, int nt, int s0);
extern "C" __global__ void k_upd_flush_small(const DChain *chains, int nch, int grp, int nt, int s0);
