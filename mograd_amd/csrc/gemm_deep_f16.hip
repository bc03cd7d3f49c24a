// Copied-tile products and Linear backwards for f16 storage.
#include "gemm_16bit_deep.h"
namespace mg {
template int launch_16bit_deep<f16_t>(const GemmArgs&, Gemm16Tile, int, int, float*, hipStream_t);
template int launch_linear_bwd_deep<f16_t>(const Gemm16Problem<f16_t>&, const Gemm16Problem<f16_t>&, Gemm16Tile, int64_t, int64_t,
                                             hipStream_t);
}  // namespace mg
