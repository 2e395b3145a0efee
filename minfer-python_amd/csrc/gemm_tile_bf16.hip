// The tiled GEMM kernel for bf16 operands.
#include "gemm_tile.h"

namespace minfer_attn {
int launch_gemm_tile_bf16(const GemmParams& p, bool nt, int tile, hipStream_t stream) { return launch_gemm_tile<BF16>(p, nt, tile, stream); }
}  // namespace minfer_attn
