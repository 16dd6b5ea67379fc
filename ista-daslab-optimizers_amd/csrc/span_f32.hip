// The spanning (one-pass) and segmented step kernels for fp32 data.
#include "ma_block.hpp"

namespace ma {

int launch_span_f32(int C, int pass, unsigned grid, int lds_bytes, hipStream_t s,
                    const FusedParams &P) {
    return launch_span<RegsF32>(C, pass, grid, lds_bytes, s, P);
}

}  // namespace ma
