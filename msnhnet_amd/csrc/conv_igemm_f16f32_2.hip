// Instantiations of the implicit-GEMM convolution kernels for f16 inputs and float outputs, part 2 (see igemmDispatch).
#include "conv_igemm.hpp"

namespace msnh {
int igemmF16F32Part2(IgemmArgs &a, int groups, int tile, hipStream_t st) { return igemmDispatch<f16, float, 2>(a, groups, tile, st); }
}
