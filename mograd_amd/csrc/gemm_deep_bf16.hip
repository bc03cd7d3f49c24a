// Copied-tile products and Linear backwards for bf16 storage.
#include "gemm_16bit_deep.h"
namespace mg {
template int launch_16bit_deep<bf16_t>(const GemmArgs&, Gemm16Tile, int, int, float*, hipStream_t);
template int launch_linear_bwd_deep<bf16_t>(const Gemm16Problem<bf16_t>&, const Gemm16Problem<bf16_t>&, Gemm16Tile, int64_t, int64_t,
                                             hipStream_t);
}  // namespace mg
