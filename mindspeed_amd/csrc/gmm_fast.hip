// One product per launch on the fast 16-bit tiles: the bf16 kernels, and the choice of the type (fp16: gmm_fast_fp16.hip).
#include "gmm_fast_kernel.h"
#ifdef MS_TRACE_TILES
#include "gmm_pair.hip"      // (the stamps of both in one array; the diagnostic library does without the unit of its own)
#endif

namespace ms {

int launch_gmm16_fast(hipStream_t stream, const GmmArgs &args, int dtype, int out_mode, bool a_red, bool b_red,
                      unsigned grid, bool lists) {
    if (dtype == MS_BF16) return launch_fast_as<MS_BF16>(stream, args, out_mode, a_red, b_red, grid, lists);
    return launch_gmm16_fast_fp16(stream, args, out_mode, a_red, b_red, grid, lists);
}

}  // namespace ms

#ifdef MS_TRACE_TILES
// Diagnostic builds only: ms_trace_clear zeroes the tile trace (call it before the launch to be looked at: records of
// earlier, larger launches would otherwise remain), ms_trace_read copies its first n values (8 per record) to host memory.
extern "C" int ms_trace_clear(void) {
    static long long zeros[ms::kTraceSlots * 8];
    if (hipDeviceSynchronize() != hipSuccess) return MS_ERR_HIP;
    return hipMemcpyToSymbol(HIP_SYMBOL(ms::g_tile_trace), zeros, sizeof(zeros)) == hipSuccess ? MS_OK : MS_ERR_HIP;
}

extern "C" int ms_trace_read(long long *host, int n) {
    if (n < 0 || n > ms::kTraceSlots * 8) return MS_ERR_INVALID_ARGUMENT;
    return hipMemcpyFromSymbol(host, HIP_SYMBOL(ms::g_tile_trace), sizeof(long long) * n) == hipSuccess ? MS_OK : MS_ERR_HIP;
}
#endif
