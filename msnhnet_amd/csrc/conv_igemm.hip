// Host side of the implicit-GEMM convolution: argument marshalling and the default tile heuristic.
#include "conv_igemm.hpp"

namespace msnh {

int igemmF16F16Part0(IgemmArgs &a, int groups, int tile, hipStream_t st);
int igemmF16F16Part1(IgemmArgs &a, int groups, int tile, hipStream_t st);
int igemmF16F16Part2(IgemmArgs &a, int groups, int tile, hipStream_t st);

int igemmF16F16(IgemmArgs &a, int groups, int tile, hipStream_t st)
{
    return tile % kIgemmParts == 0 ? igemmF16F16Part0(a, groups, tile, st) : (tile % kIgemmParts == 1 ? igemmF16F16Part1(a, groups, tile, st) : igemmF16F16Part2(a, groups, tile, st));
}

int igemmF16F32Part0(IgemmArgs &a, int groups, int tile, hipStream_t st);
int igemmF16F32Part1(IgemmArgs &a, int groups, int tile, hipStream_t st);
int igemmF16F32Part2(IgemmArgs &a, int groups, int tile, hipStream_t st);

int igemmF16F32(IgemmArgs &a, int groups, int tile, hipStream_t st)
{
    return tile % kIgemmParts == 0 ? igemmF16F32Part0(a, groups, tile, st) : (tile % kIgemmParts == 1 ? igemmF16F32Part1(a, groups, tile, st) : igemmF16F32Part2(a, groups, tile, st));
}

int igemmF32F32Part0(IgemmArgs &a, int groups, int tile, hipStream_t st);
int igemmF32F32Part1(IgemmArgs &a, int groups, int tile, hipStream_t st);
int igemmF32F32Part2(IgemmArgs &a, int groups, int tile, hipStream_t st);

int igemmF32F32(IgemmArgs &a, int groups, int tile, hipStream_t st)
{
    return tile % kIgemmParts == 0 ? igemmF32F32Part0(a, groups, tile, st) : (tile % kIgemmParts == 1 ? igemmF32F32Part1(a, groups, tile, st) : igemmF32F32Part2(a, groups, tile, st));
}


// Default tile: BM follows the output-channel count so narrow layers do not waste MFMA rows; deep K
// (>= 8 vectors per tap) moves 8 vectors per row per step, shallow K 4.
int igemmHeuristicTile(const msnh_conv_desc *d)
{
    const int vec = d->dtype == MSNH_F16 ? 8 : 4;
    const int cinG = d->in_c / d->groups, coutG = d->out_c / d->groups;
    const bool deep = cinG >= 8 * vec;
    if (coutG <= 32) return deep ? 5 : 6;
    if (coutG <= 64) return deep ? 3 : 4;
    return deep ? 1 : 2;
}

int igemmTileCount() { return kIgemmTiles; }
int igemmTailTileFirst() { return kIgemmTailTileFirst; }

int igemmSlicedTiles(int *tiles, int cap)
{
    const int n = static_cast<int>(sizeof(kIgemmSlicedTiles) / sizeof(kIgemmSlicedTiles[0]));
    for (int i = 0; i < n && i < cap; ++i) tiles[i] = kIgemmSlicedTiles[i];
    return n;
}

size_t igemmSplitKWorkspaceBytes(const msnh_conv_desc *d)
{
    return static_cast<size_t>(kSplitKMax) * d->batch * d->out_h * d->out_w * d->out_c * sizeof(float);
}

// MSNH_CONV_IGEMM_SPLITK (callers of the C interface; the plans use the sum inside the launch): the kernel with float32 results writes the raw partial sums
// of its slices, slicePitch apart, and a second launch sums them in slice order (so the result does not depend on timing) and applies the
// convolution's epilogue.  One thread per (pixel, 4 channels).
template <typename T, typename TOut>
__global__ __launch_bounds__(256) void splitKReduceKernel(IgemmArgs a, int outC, long long total)
{
    const long long idx = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= total) return;
    const int cq = outC / 4;
    const int c = static_cast<int>(idx % cq) * 4;
    const long long p = idx / cq;
    const float *w = a.ws + static_cast<size_t>(p) * a.wsLd + c;
    f32x4 acc = *reinterpret_cast<const f32x4 *>(w);
    for (int s = 1; s < a.splitK; ++s) acc += *reinterpret_cast<const f32x4 *>(w + static_cast<size_t>(s) * a.P * a.wsLd);
    const T *res = static_cast<const T *>(a.res);
    TOut *y = static_cast<TOut *>(a.y);
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        const float sc = a.scale ? a.scale[c + k] : 1.f;
        const float sh = a.shift ? a.shift[c + k] : 0.f;
        float v = activate(acc[k] * sc + sh, a.act, a.actParam);
        if (a.hasRes) v = activate(v + a.resMul * toF(res[static_cast<size_t>(p) * a.resLd + c + k]), a.act2, a.act2Param);
        y[static_cast<size_t>(p) * a.outLd + c + k] = fromF<TOut>(a.outMul * v);
    }
}

static int convIgemmSplitK(IgemmArgs &a, const msnh_conv_desc *d, int tile, hipStream_t st)
{
    IgemmArgs e = a;
    e.scale = e.shift = nullptr;
    e.act = MSNH_ACT_NONE; e.hasRes = 0; e.res = nullptr; e.outMul = 1.f;
    e.y = a.ws;
    e.outLd = a.wsLd;
    e.slicePitch = static_cast<size_t>(a.P) * a.wsLd;
    e.vecOk = (a.wsLd % 8 == 0) && (a.coutG % 8 == 0 || d->groups == 1);
    const int rc = d->dtype != MSNH_F16 ? igemmF32F32(e, d->groups, tile, st) : igemmF16F32(e, d->groups, tile, st);
    if (rc != 0 || a.dryRun) return rc;
    a.splitK = e.splitK;
    const long long total = static_cast<long long>(a.P) * (d->out_c / 4);
    const auto kern = d->dtype != MSNH_F16 ? splitKReduceKernel<float, float> : (d->out_dtype == MSNH_F16 ? splitKReduceKernel<f16, f16> : splitKReduceKernel<f16, float>);
    hipLaunchKernelGGL(kern, dim3(gridFor(total, 256)), dim3(256), 0, st, a, d->out_c, total);
    MSNH_LAUNCH_CHECK();
    return 0;
}

// tail != nullptr: the launch also computes the 1x1 convolution described there (msnh_hip_conv2d_tail); d->tile then names one of the
// tiles that carry a tail, 0 the first of them that takes the shape.
static int convIgemmAny(const msnh_conv_desc *d, const void *x, const void *w, const float *scale, const float *shift,
                        const void *residual, void *y, hipStream_t st, bool dryRun, void *splitWs, size_t splitWsBytes,
                        const msnh_conv_tail_desc *tail, const void *w2, const float *scale2, const float *shift2, void *z, size_t *wsNeed = nullptr,
                        const msnh_conv_pair_desc *pair = nullptr)
{
    IgemmArgs a;
    a.tailOn = tail ? 1 : 0;
    a.w2 = w2; a.scale2 = scale2; a.shift2 = shift2; a.z = z;
    a.cout2 = tail ? tail->out_c : 0; a.zLd = tail ? tail->out_ld : 0; a.act3 = tail ? tail->act : MSNH_ACT_NONE; a.writeY = tail ? (tail->write_y ? 1 : 0) : 1;
    a.act3Param = tail ? tail->act_param : 0.f; a.zMul = tail ? tail->out_mul : 1.f;
    a.w2Bytes = tail ? static_cast<unsigned>(tail->out_c) * static_cast<unsigned>(d->out_c) * 2u : 0u;
    a.pairC = 0;
    if (pair)
    {
        a.pairC = pair->first_c; a.z = z; a.zLd = pair->out_ld2; a.act3 = pair->act; a.act3Param = pair->act_param; a.zMul = pair->out_mul;
    }
    a.x = x; a.w = w; a.scale = scale; a.shift = shift; a.res = residual; a.y = y;
    a.batch = d->batch; a.H = d->in_h; a.W = d->in_w; a.inLd = d->in_ld;
    a.OH = d->out_h; a.OW = d->out_w; a.outLd = d->out_ld; a.resLd = d->res_ld;
    a.cinG = d->in_c / d->groups; a.coutG = d->out_c / d->groups;
    a.taps = d->ksize * d->ksize; a.ksize = d->ksize; a.stride = d->stride; a.pad = d->pad; a.dil = d->dilation;
    a.P = d->batch * d->out_h * d->out_w;
    a.up2 = d->out_upsample == 2 ? 1 : 0;
    a.xcdGm = d->xcd_blocks;
    a.yBytes = a.up2 ? static_cast<unsigned>(static_cast<unsigned long long>(d->batch) * d->out_h * d->out_w * 4ull * d->out_ld * dtypeSize(d->out_dtype)) : 0u;
    a.byOW = makeFastDiv(static_cast<unsigned>(d->out_w));
    a.byOH = makeFastDiv(static_cast<unsigned>(d->out_h));
    a.byKsize = makeFastDiv(static_cast<unsigned>(d->ksize));
    a.tapRows = 0;
    if (a.taps <= 64) for (int q = 0; q < d->ksize; ++q) a.tapRows |= 1ull << (q * d->ksize);      // (more taps are refused)
    a.pointwise = d->ksize == 1 && d->stride == 1 && d->pad == 0 ? 1 : 0;
    a.patchOk = (d->ksize == 3 && d->stride == 1 && d->pad == 1 && d->dilation == 1 && d->groups == 1 && d->out_h == d->in_h && d->out_w == d->in_w) ? 1 : 0;
    a.patchRows = 0; a.mTiles = 0; a.cChunks = 0; a.nIter = 0;
    a.dryRun = dryRun ? 1 : 0;
    {
        const unsigned long long es = dtypeSize(d->dtype);
        const unsigned long long xb = ((static_cast<unsigned long long>(d->batch) * d->in_h * d->in_w - 1) * d->in_ld + d->in_c) * es;
        const unsigned long long wb = static_cast<unsigned long long>(d->out_c) * a.taps * a.cinG * es;
        a.buffersOk = xb < 0x7fffffffull && wb < 0x7fffffffull;
        a.xBytes = static_cast<unsigned>(xb);
        a.wBytes = static_cast<unsigned>(wb);
        a.ragged = 0;
    }
    a.act = d->act; a.act2 = d->act2; a.hasRes = (d->has_residual && residual) ? 1 : 0;
    a.actParam = d->act_param; a.act2Param = d->act2_param; a.resMul = d->res_mul; a.outMul = d->out_mul;
    const size_t outEl = dtypeSize(d->out_dtype);
    // 8-channel vector stores / residual loads need 8-element alignment of every row start
    a.vecOk = (d->out_ld % 8 == 0) && ((d->out_c / d->groups) % 8 == 0 || d->groups == 1) &&
              (reinterpret_cast<uintptr_t>(y) % (8 * outEl) == 0) &&
              (!a.hasRes || (d->res_ld % 8 == 0 && reinterpret_cast<uintptr_t>(residual) % 16 == 0));
    if (pair) a.vecOk = a.vecOk && pair->out_ld2 % 8 == 0 && reinterpret_cast<uintptr_t>(z) % (8 * outEl) == 0;
    a.splitMax = 0; a.splitK = 1; a.fusedK = 0; a.wsNeed = a.wsBytes = 0; a.ws = nullptr; a.wsLd = d->out_c; a.slicePitch = 0;
    if (a.up2) MSNH_REQUIRE(d->algo != MSNH_CONV_IGEMM_SPLITK && !tail, "conv2d: the upsampling epilogue goes with the plain implicit GEMM");
    if (d->algo == MSNH_CONV_IGEMM_SPLITK)
    {
        MSNH_REQUIRE(d->out_c % 4 == 0, "conv2d: split-K needs out_c to be a multiple of 4");
        if (!dryRun)
        {
            MSNH_REQUIRE(splitWs && reinterpret_cast<uintptr_t>(splitWs) % 16 == 0 && splitWsBytes >= igemmSplitKWorkspaceBytes(d),
                         "conv2d: split-K needs a 16-byte aligned workspace of msnh_hip_conv2d_workspace_bytes() bytes");
        }
        a.splitMax = kSplitKMax;
        a.ws = static_cast<float *>(splitWs);
    }
    int tile = d->tile;
    if (d->algo == MSNH_CONV_IGEMM_FUSEDK)
    {
        a.fusedK = d->tile >> 8;
        tile = d->tile & 255;
        MSNH_REQUIRE(!tail && tile >= 1 && tile <= kIgemmTiles && a.fusedK >= 2 && a.fusedK <= 32, "conv2d: IGEMM_FUSEDK takes desc.tile = tile + 256 * slices, 2 to 32 slices");
        MSNH_REQUIRE(dryRun || reinterpret_cast<uintptr_t>(splitWs) % 16 == 0, "conv2d: the workspace must be 16-byte aligned");
        a.ws = static_cast<float *>(splitWs);
        a.wsBytes = splitWsBytes;
    }
    if (tail)
    {
        MSNH_REQUIRE(d->dtype == MSNH_F16 && d->out_dtype == MSNH_F16 && d->groups == 1 && d->algo != MSNH_CONV_IGEMM_SPLITK, "conv2d_tail: float16, ungrouped, unsplit");
        if (tile <= 0) tile = d->out_c > 128 ? kIgemmTailTileFirst : kIgemmTailTileFirst + 1;
        MSNH_REQUIRE(tile >= kIgemmTailTileFirst && tile <= kIgemmTiles, "conv2d_tail: tile %d carries no tail", tile);
        if (!dryRun)
            MSNH_REQUIRE(reinterpret_cast<uintptr_t>(z) % 16 == 0 && reinterpret_cast<uintptr_t>(w2) % 16 == 0, "conv2d_tail: z and w2 must be 16-byte aligned");
        else a.vecOk = (d->out_ld % 8 == 0) && (d->out_c % 8 == 0) && (!d->has_residual || d->res_ld % 8 == 0);
    }
    if (tile <= 0 || tile > kIgemmTiles) tile = igemmHeuristicTile(d);
    MSNH_REQUIRE(d->dtype == MSNH_F16 || d->out_dtype == MSNH_F32, "igemm: float32 input needs float32 output");
    if (a.splitMax > 1) return convIgemmSplitK(a, d, tile, st);
    const int rc = d->dtype != MSNH_F16 ? igemmF32F32(a, d->groups, tile, st)
                                        : (d->out_dtype == MSNH_F16 ? igemmF16F16(a, d->groups, tile, st) : igemmF16F32(a, d->groups, tile, st));
    if (wsNeed) *wsNeed = a.wsNeed;
    return rc;
}

int convIgemmWs(const msnh_conv_desc *d, const void *x, const void *w, const float *scale, const float *shift,
                const void *residual, void *y, hipStream_t st, bool dryRun, void *splitWs, size_t splitWsBytes)
{
    return convIgemmAny(d, x, w, scale, shift, residual, y, st, dryRun, splitWs, splitWsBytes, nullptr, nullptr, nullptr, nullptr, nullptr);
}

// Workspace of a sliced launch as desc.tile describes it; 0: the shape and tile do not take it.
size_t igemmFusedKWorkspaceBytes(const msnh_conv_desc *d)
{
    size_t need = 0;
    msnh_conv_desc t = *d;
    t.algo = MSNH_CONV_IGEMM_FUSEDK;
    return convIgemmAny(&t, d, d, nullptr, nullptr, nullptr, &t, nullptr, true, nullptr, 0, nullptr, nullptr, nullptr, nullptr, nullptr, &need) == 0 ? need : 0;
}

int convIgemmTail(const msnh_conv_desc *d, const msnh_conv_tail_desc *tail, const void *x, const void *w, const float *scale, const float *shift,
                  const void *residual, void *y, const void *w2, const float *scale2, const float *shift2, void *z, hipStream_t st, bool dryRun)
{
    return convIgemmAny(d, x, w, scale, shift, residual, y, st, dryRun, nullptr, 0, tail, w2, scale2, shift2, z);
}

// d->out_ld: the first tensor's.  Tile 0: the one that the shape's rule names, whose wave tiles have 64 channels, or, where the border between the tensors cuts
// those, a 64 x 64 tile, whose wave tiles have 32.  (Of the tiles with 32, float32 1x1 512 -> 256 at 38 x 38, one / eight images: 64 x 64 13.3 / 30.5 us, 64 x 128
// 20.4 / 41.4, 32 x 256 21.1 / 42.8, 128 x 192 39.7 / 44.8; float16 256 -> 256 at 38 x 38, eight images, 64 x 64 7.0, 128 x 192 7.9.)
int convIgemmPair(const msnh_conv_desc *d, const msnh_conv_pair_desc *pair, const void *x, const void *w, const float *scale, const float *shift, void *y, void *y2,
                  hipStream_t st, bool dryRun, void *ws, size_t wsBytes)
{
    msnh_conv_desc c = *d;
    if (c.algo != MSNH_CONV_IGEMM_FUSEDK && c.tile == 0 && pair->first_c % 64 != 0) c.tile = c.in_c >= (c.dtype == MSNH_F16 ? 64 : 32) ? 12 : 6;
    return convIgemmAny(&c, x, w, scale, shift, nullptr, y, st, dryRun, ws, wsBytes, nullptr, nullptr, nullptr, nullptr, y2, nullptr, pair);
}

int convIgemm(const msnh_conv_desc *d, const void *x, const void *w, const float *scale, const float *shift,
              const void *residual, void *y, hipStream_t st, bool dryRun)
{
    return convIgemmWs(d, x, w, scale, shift, residual, y, st, dryRun, nullptr, 0);
}

} // namespace msnh
