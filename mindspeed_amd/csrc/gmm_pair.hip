// Both gradients of one grouped matmul in one launch on the fast 16-bit tiles (gmm_fast_tile.h): dX, both operands contiguous
// along the reduction dim, and dW, neither.  The form with tables and a 16-bit dW keeps four
// registers in scratch through the last K step, one store and one load per tile; the K loops have none.
#include "gmm_fast_tile.h"

namespace ms {
namespace {

template <int DT, bool RED, int OUT, bool DIRECT>
__device__ __forceinline__ void pair_tile(const GmmArgs &p, int b, char *lds) {
    TileCoord tc;
    if constexpr (DIRECT) tc = tile_from_list<!RED>(p, b);
    else tc = locate_tile<true, RED>(p.table, b);
    if (!tc.valid) return;
    MS_TRACE(2);
    if (tc.tile_rows == 256) gmm16_tile<DT, RED, RED, OUT, 256>(p, tc, lds);
    else if (tc.tile_rows == 128) gmm16_tile<DT, RED, RED, OUT, 128>(p, tc, lds);
    else gmm16_tile<DT, RED, RED, OUT, 64>(p, tc, lds);
    MS_TRACE_END(tc.tile_rows, !RED);
}

template <int DT, int OUT, bool DIRECT>
__global__ __launch_bounds__(256) void gmm16_pair_kernel(const GmmArgs dx, const GmmArgs dw, int first, int dw_first) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    MS_TRACE(1);
    const int b = blockIdx.x;
    const bool second = b >= first;
    const int own = second ? b - first : b;
    if (second == (dw_first == 0)) pair_tile<DT, false, OUT, DIRECT>(dw, own, lds);
    else pair_tile<DT, true, OUT_SAME, DIRECT>(dx, own, lds);
}

template <int DT, int OUT>
const void *pick(bool direct) {
    return direct ? reinterpret_cast<const void *>(&gmm16_pair_kernel<DT, OUT, true>)
                  : reinterpret_cast<const void *>(&gmm16_pair_kernel<DT, OUT, false>);
}

}  // namespace

int launch_gmm16_pair(hipStream_t stream, const GmmArgs &dx, unsigned dx_grid, const GmmArgs &dw, unsigned dw_grid, int dtype,
                      int out_mode, bool dw_first, bool direct) {
    const void *fn = dtype == MS_BF16 ? (out_mode == ACC_F32 ? pick<MS_BF16, ACC_F32>(direct) : pick<MS_BF16, OUT_SAME>(direct))
                                      : (out_mode == ACC_F32 ? pick<MS_FP16, ACC_F32>(direct) : pick<MS_FP16, OUT_SAME>(direct));
    hipError_t e = set_max_dynamic_lds(fn, kDmaBytes);
    MS_REQUIRE(e == hipSuccess, MS_ERR_HIP, "ms_gmm: hipFuncSetAttribute: %s", hipGetErrorString(e));
    GmmArgs args[2] = {dx, dw};
    int first = static_cast<int>(dw_first ? dw_grid : dx_grid), order = dw_first ? 1 : 0;
    void *kargs[] = {&args[0], &args[1], &first, &order};
    e = hipLaunchKernel(fn, dim3(dx_grid + dw_grid), dim3(256), kargs, kDmaBytes, stream);
    MS_REQUIRE(e == hipSuccess, MS_ERR_HIP, "ms_gmm: launch failed: %s", hipGetErrorString(e));
    return MS_OK;
}

}  // namespace ms
