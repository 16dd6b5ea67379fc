// The fused block kernels for bf16 data with longer windows (update_long).
#include "ma_block.hpp"

namespace ma {

int launch_fused_long_bf16(int C, unsigned grid, int lds_bytes, hipStream_t s,
                           const FusedParams &P) {
    return launch_fused_long<RegsBF16>(C, grid, lds_bytes, s, P);
}

}  // namespace ma
