// Instantiations of the implicit-GEMM convolution kernels for f16 inputs and f16 outputs, part 1 (see igemmDispatch).
#include "conv_igemm.hpp"

namespace msnh {
int igemmF16F16Part1(IgemmArgs &a, int groups, int tile, hipStream_t st) { return igemmDispatch<f16, f16, 1>(a, groups, tile, st); }
}
