// Instantiations of the implicit-GEMM convolution kernels for float inputs and float outputs, part 0 (see igemmDispatch).
#include "conv_igemm.hpp"

namespace msnh {
int igemmF32F32Part0(IgemmArgs &a, int groups, int tile, hipStream_t st) { return igemmDispatch<float, float, 0>(a, groups, tile, st); }
}
