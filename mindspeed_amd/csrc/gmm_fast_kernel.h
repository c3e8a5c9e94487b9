// One product per launch on the fast tiles (gmm_fast_tile.h): the kernel and its launch, for one data type per translation unit.
#pragma once

#include "gmm_fast_tile.h"

namespace ms {
namespace {

// LISTS: the launch may come with per-XCD lists of entries.  Always so for the split on rows (A_RED); the weight-gradient
// product has a variant of its own for launches of many groups, so that the common one does not carry that lookup.
// DIRECT: tiles are found from the group list.  Kernels of their own too: the code for it merely present beside the table's
// cost long forward launches 1.1 to 1.6 % (8 experts x 4096 x 28672 1554 -> 1571 us, 64 x 2048 x 2816 712 -> 724).
template <int DT, bool A_RED, bool B_RED, int OUT, bool LISTS = A_RED, bool DIRECT = false>
__global__ __launch_bounds__(256) void gmm16_fast_kernel(const GmmArgs p) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    MS_TRACE(1);
    TileCoord tc;
    if constexpr (DIRECT) tc = tile_from_list<!A_RED>(p, blockIdx.x);
    else tc = locate_tile<LISTS, A_RED>(p.table, blockIdx.x);
    if (!tc.valid) return;
    MS_TRACE(2);
    if (tc.tile_rows == 256) {
        gmm16_tile<DT, A_RED, B_RED, OUT, 256>(p, tc, lds);
    } else if (OUT == OUT_SAME && A_RED && tc.e.split != 0) {
        // one part of a small tail tile whose reduction is split: fp32 partial sums into the split workspace
        // (rows of `cols` floats; the entry's c_off leads to this part's block)
        GmmArgs q = p;
        q.c = p.split_ws;
        q.c_stride_row = p.cols;
        if (tc.tile_rows == 128) gmm16_tile<DT, A_RED, B_RED, OUT_F32, 128>(q, tc, lds);
        else gmm16_tile<DT, A_RED, B_RED, OUT_F32, 64>(q, tc, lds);
    } else if (tc.tile_rows == 128) {
        gmm16_tile<DT, A_RED, B_RED, OUT, 128>(p, tc, lds);
    } else {
        gmm16_tile<DT, A_RED, B_RED, OUT, 64>(p, tc, lds);
    }
    MS_TRACE_END(tc.tile_rows, !A_RED);
}

template <int DT, int OUT>
int launch_fast(hipStream_t stream, const GmmArgs &args, bool a_red, bool b_red, unsigned grid, bool lists) {
    const void *fn;
    const bool direct = args.group_list != nullptr;
    auto pick = [&](const void *from_list, const void *from_table) { return direct ? from_list : from_table; };
    MS_REQUIRE(a_red || !b_red, MS_ERR_UNSUPPORTED, "ms_gmm: operand layout not supported");   // (the caller keeps it off this path)
    if constexpr (OUT == OUT_SWIGLU) {
        MS_REQUIRE(a_red && !b_red, MS_ERR_UNSUPPORTED, "ms_gmm_swiglu: operand layout not supported");
        fn = pick(reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, true, false, OUT, false, true>),
                  reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, true, false, OUT>));
    } else if constexpr (OUT == OUT_SWIGLU_GRAD) {
        MS_REQUIRE(a_red && b_red, MS_ERR_UNSUPPORTED, "ms_gmm_swiglu_grad: operand layout not supported");
        fn = pick(reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, true, true, OUT, false, true>),
                  reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, true, true, OUT>));
    } else if (a_red && b_red) {
        fn = pick(reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, true, true, OUT, false, true>),
                  reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, true, true, OUT>));
    } else if (a_red) {
        fn = pick(reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, true, false, OUT, false, true>),
                  reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, true, false, OUT>));
    } else if (direct) fn = reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, false, false, OUT, false, true>);
    else if (lists) fn = reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, false, false, OUT, true>);
    else fn = reinterpret_cast<const void *>(&gmm16_fast_kernel<DT, false, false, OUT>);
    hipError_t e = set_max_dynamic_lds(fn, kDmaBytes);
    MS_REQUIRE(e == hipSuccess, MS_ERR_HIP, "ms_gmm: hipFuncSetAttribute: %s", hipGetErrorString(e));
    GmmArgs copy = args;
    void *kargs[] = {&copy};
    e = hipLaunchKernel(fn, dim3(grid), dim3(256), kargs, kDmaBytes, stream);
    MS_REQUIRE(e == hipSuccess, MS_ERR_HIP, "ms_gmm: launch failed: %s", hipGetErrorString(e));
    return MS_OK;
}

template <int DT>
int launch_fast_as(hipStream_t stream, const GmmArgs &args, int out_mode, bool a_red, bool b_red, unsigned grid, bool lists) {
    switch (out_mode) {
        case OUT_SWIGLU: return launch_fast<DT, OUT_SWIGLU>(stream, args, a_red, b_red, grid, lists);
        case OUT_SWIGLU_GRAD: return launch_fast<DT, OUT_SWIGLU_GRAD>(stream, args, a_red, b_red, grid, lists);
        case OUT_SAME: return launch_fast<DT, OUT_SAME>(stream, args, a_red, b_red, grid, lists);
        case OUT_F32: return launch_fast<DT, OUT_F32>(stream, args, a_red, b_red, grid, lists);
        default: return launch_fast<DT, ACC_F32>(stream, args, a_red, b_red, grid, lists);
    }
}

}  // namespace
}  // namespace ms
