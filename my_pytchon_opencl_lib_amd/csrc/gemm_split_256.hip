// gemm_split_kernel instantiations for 256 tiles (kernel: gemm_split.h, gemm_split.hip).
#include "gemm_split.h"

namespace migemm {

int launch_split_256(hipStream_t stream, TiledArgs &a, bool akc, bool bkc) {
    return launch_split_layouts<256, 256, 4, 2>(stream, a, akc, bkc);
}

}  // namespace migemm
