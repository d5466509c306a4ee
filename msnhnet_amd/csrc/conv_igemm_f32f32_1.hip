// Instantiations of the implicit-GEMM convolution kernels for float inputs and float outputs, part 1 (see igemmDispatch).
#include "conv_igemm.hpp"

namespace msnh {
int igemmF32F32Part1(IgemmArgs &a, int groups, int tile, hipStream_t st) { return igemmDispatch<float, float, 1>(a, groups, tile, st); }
}
