// One product per launch on the fast 16-bit tiles: the fp16 kernels.
#include "gmm_fast_kernel.h"

namespace ms {

int launch_gmm16_fast_fp16(hipStream_t stream, const GmmArgs &args, int out_mode, bool a_red, bool b_red, unsigned grid, bool lists) {
    return launch_fast_as<MS_FP16>(stream, args, out_mode, a_red, b_red, grid, lists);
}

}  // namespace ms
