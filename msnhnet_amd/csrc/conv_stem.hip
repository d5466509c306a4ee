// First-layer convolution on the matrix cores: 3x3 / 5x5 / 7x7 filter over <= 4 input channels, and the 6x6 stride-2 filter of the focus opening
// (7x7 and 6x6 over 3 channels have a kernel of their own further down), read straight from
// the NCHW float32 network input (layout conversion and cast to float16 fused), NHWC float16 out.
//
// GEMM view: all output channels (32, 64 or 128) x 32 consecutive output pixels of one row per wavefront,
// K = ksize^2 * Cin padded to a multiple of 32, two 32x32x16 MFMAs per 32 of K and 32 channels.  The kernel is
// bound by the write of the output and by the scalar gathers (16 per lane and 32 of K) that assemble the B
// operand; where each K index points inside the image is a table in the kernel-argument segment, read with scalar
// loads.  The weights (operand A, already in MFMA lane order) and the channel affine sit in LDS.
//
// The rows of the MFMA are a permutation of the channels: MFMA row 8q + 4h + e computes channel 16h + 4q + e.
// The 32x32 accumulator layout gives lane l, register r the row 8(r/4) + 4(l/32) + r%4, so with that permutation
// the 16 registers of a lane are 16 CONSECUTIVE channels of its pixel: two 16-byte stores, no transposition.
#include "common.hpp"
#include <type_traits>

namespace msnh {

namespace {

template <int I, int N, typename F> __device__ __forceinline__ void staticFor(F &&f)
{
    if constexpr (I < N)
    {
        f(std::integral_constant<int, I>());
        staticFor<I + 1, N>(f);
    }
}

typedef unsigned stemU32x4 __attribute__((ext_vector_type(4)));

constexpr int kStemMaxK = 160;          // 7x7x3 = 147 padded to five 32-wide K blocks

struct StemArgs
{
    const float *x;
    const f16   *wA;        // [mBlocks][KB*2][64 lanes][8]
    const float *scale;
    const float *shift;
    f16         *y;
    int B, H, W, OH, OW, outLd, outC, stride, pad, cin, ksize;
    int groupsPerRow;       // ceil(OW / 32)
    int nGroups;            // B * OH * groupsPerRow
    int act;
    float actParam, outMul;
    // per K index: offset of the tap inside one batch item's NCHW planes (ci*H*W + ky*W + kx), and ky << 8 | kx.
    // Lives in the kernel-argument segment: the kernel indexes it with compile-time constants, i.e. scalar loads.
    int koff[kStemMaxK];
    int kyx[kStemMaxK];     // ky << 8 | kx; K padding: ky = 32767 (never inside the image)
};

// operand B of 16 K indices (8 per half of the wavefront) with everything from the K-th on set to zero
template <int K> __device__ __forceinline__ f16x8 stemKeepTaps(f16x8 b, bool hi)
{
    stemU32x4 v = __builtin_bit_cast(stemU32x4, b);
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const unsigned lo = (2 * j < K ? 0xffffu : 0u) | (2 * j + 1 < K ? 0xffff0000u : 0u), up = (2 * j + 8 < K ? 0xffffu : 0u) | (2 * j + 9 < K ? 0xffff0000u : 0u);
        if (lo != ~0u || up != ~0u) v[j] &= hi ? up : lo;
    }
    return __builtin_bit_cast(f16x8, v);
}

// TAPS: ksize^2 * Cin, in KB 32-wide K blocks; MBLK: 32-channel output blocks.  What fills the last block up has zero weights, but zero times an
// infinite pixel is not zero: its operand is blanked too, by masks that the number of taps makes constants (a mask per dword that holds padding; as
// kernel arguments they cost 3 us of 4 for MobileNetV2's first layer, one image, computed in the kernel 3 % of 28 at batch 64).
template <int TAPS, int MBLK>
__global__ __launch_bounds__(256) void convStemMfmaKernel(StemArgs a)
{
    touchArgs(a);
    constexpr int KB = (TAPS + 31) / 32;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    f16 *wl = reinterpret_cast<f16 *>(smem);                                  // [MBLK][KB*2][64][8]
    float *ssl = reinterpret_cast<float *>(smem + MBLK * KB * 2 * 1024);       // [2][MBLK*32]
    for (int i = threadIdx.x; i < MBLK * KB * 2 * 64; i += 256)
        reinterpret_cast<f16x8 *>(wl)[i] = reinterpret_cast<const f16x8 *>(a.wA)[i];
    for (int i = threadIdx.x; i < MBLK * 32; i += 256)
    {
        ssl[i] = a.scale && i < a.outC ? a.scale[i] : 1.f;
        ssl[MBLK * 32 + i] = a.shift && i < a.outC ? a.shift[i] : 0.f;
    }
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int n = lane & 31;
    const bool hi = lane >= 32;
    // A workgroup takes one contiguous run of pixel groups (its four wavefronts interleaved), and the hardware's round-robin of
    // workgroup ids over the 8 XCDs is undone so that an XCD works on one contiguous run of image rows: the input rows that
    // neighbouring output rows share are then read from memory once, not once per XCD that happens to need them.
    const int nBlocks = static_cast<int>(gridDim.x);
    const int perXcd = (nBlocks + 7) / 8;
    const int logical = static_cast<int>(blockIdx.x % 8) * perXcd + static_cast<int>(blockIdx.x / 8);
    const int perBlock = (a.nGroups + nBlocks - 1) / nBlocks;
    const int gBegin = logical < nBlocks ? logical * perBlock : a.nGroups;
    const int gEnd = min(a.nGroups, gBegin + perBlock);
    const int planes = a.cin * a.H * a.W;

    const bool lin = (a.act == MSNH_ACT_LEAKY || a.act == MSNH_ACT_RELU || a.act == MSNH_ACT_NONE);
    const float slope = a.act == MSNH_ACT_LEAKY ? a.actParam : (a.act == MSNH_ACT_RELU ? 0.f : 1.f);

    for (int g = gBegin + static_cast<int>(threadIdx.x >> 6); g < gEnd; g += 4)
    {
        const int gx = g % a.groupsPerRow;
        const int row = g / a.groupsPerRow;
        const int oy = row % a.OH;
        const int b = row / a.OH;
        const int ox = gx * 32 + n;
        const int iy0 = oy * a.stride - a.pad;
        const int ix0 = ox * a.stride - a.pad;
        // valid taps are dereferenced only; the base may lie outside the tensor
        const float *xb = a.x + static_cast<long long>(b) * planes + static_cast<long long>(iy0) * a.W + ix0;
        f32x16 acc[MBLK];
#pragma unroll
        for (int mb = 0; mb < MBLK; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;

        // wave-uniform: every tap of every pixel of the group lies inside the image (no bounds tests then)
        const int ixFirst = gx * 32 * a.stride - a.pad;
        const int ixLast  = (gx * 32 + 31) * a.stride - a.pad;
        const bool interior = iy0 >= 0 && iy0 + a.ksize <= a.H && ixFirst >= 0 && ixLast + a.ksize <= a.W && gx * 32 + 31 < a.OW;
        staticFor<0, KB>([&](auto kbTag) {
            constexpr int kb = decltype(kbTag)::value;
            float v[16];
            if (interior)
            {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                {
                    // lanes 0-31 hold K index kLo, lanes 32-63 kLo + 8; K padding has offset 0, its value is blanked below
                    const int kLo = kb * 32 + (i / 8) * 16 + (i % 8);
                    v[i] = kLo >= TAPS ? 0.f : xb[hi ? a.koff[kLo + 8] : a.koff[kLo]];
                }
            }
            else
            {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                {
                    const int kLo = kb * 32 + (i / 8) * 16 + (i % 8);
                    const int off = hi ? a.koff[kLo + 8] : a.koff[kLo];
                    const int yx  = hi ? a.kyx[kLo + 8] : a.kyx[kLo];
                    const unsigned iy = static_cast<unsigned>(iy0 + (yx >> 8)), ix = static_cast<unsigned>(ix0 + (yx & 255));
                    v[i] = (iy < static_cast<unsigned>(a.H) && ix < static_cast<unsigned>(a.W)) ? xb[off] : 0.f;
                }
            }
            f16x8 b0, b1;
#pragma unroll
            for (int e = 0; e < 8; ++e) { b0[e] = static_cast<f16>(v[e]); b1[e] = static_cast<f16>(v[8 + e]); }
            if constexpr (kb == KB - 1)
            {
                b0 = stemKeepTaps<TAPS - kb * 32>(b0, hi);
                b1 = stemKeepTaps<TAPS - kb * 32 - 16>(b1, hi);
            }
#pragma unroll
            for (int mb = 0; mb < MBLK; ++mb)
            {
                const f16x8 wa0 = *reinterpret_cast<const f16x8 *>(wl + ((static_cast<size_t>(mb) * KB * 2 + kb * 2 + 0) * 64 + lane) * 8);
                const f16x8 wa1 = *reinterpret_cast<const f16x8 *>(wl + ((static_cast<size_t>(mb) * KB * 2 + kb * 2 + 1) * 64 + lane) * 8);
                acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wa0, b0, acc[mb], 0, 0, 0);
                acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wa1, b1, acc[mb], 0, 0, 0);
            }
        });
        if (ox < a.OW && (!hi || a.outC > 16))
        {
            f16 *yp = a.y + (static_cast<size_t>(row) * a.OW + ox) * a.outLd + (hi ? 16 : 0);
#pragma unroll
            for (int mb = 0; mb < MBLK; ++mb)
            {
                const float *scp = ssl + mb * 32 + (hi ? 16 : 0);
                const float *shp = scp + MBLK * 32;
                f16x8 o0, o1;
                float t[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) t[r] = acc[mb][r] * scp[r] + shp[r];
                if (lin)
                {
#pragma unroll
                    for (int r = 0; r < 16; ++r) t[r] = t[r] > 0.f ? t[r] : slope * t[r];
                }
                else activateArray<16>(t, a.act, a.actParam);       // one choice of the activation for the 16 values
#pragma unroll
                for (int r = 0; r < 16; ++r)
                {
                    const float u = t[r] * a.outMul;
                    if (r < 8) o0[r] = static_cast<f16>(u); else o1[r - 8] = static_cast<f16>(u);
                }
                *reinterpret_cast<f16x8 *>(yp + mb * 32) = o0;
                *reinterpret_cast<f16x8 *>(yp + mb * 32 + 8) = o1;
            }
        }
    }
}

template <int TAPS, int MBLK>
int launchStem(const StemArgs &a, unsigned blocks, hipStream_t st)
{
    constexpr int KB = (TAPS + 31) / 32;
    const size_t smem = static_cast<size_t>(MBLK) * KB * 2 * 1024 + 2 * MBLK * 32 * sizeof(float);
    auto kern = convStemMfmaKernel<TAPS, MBLK>;
    if (const int rc = allowLds(reinterpret_cast<const void *>(kern), smem)) return rc;
    hipLaunchKernelGGL(kern, dim3((blocks + 7) / 8 * 8), dim3(256), smem, st, a);      // a multiple of 8: the XCD regrouping is a bijection then
    MSNH_LAUNCH_CHECK();
    return 0;
}

// ---- 7x7 and 6x6 filters over 3 channels (the ResNet stems, the focus opening): K ordered by image rows ----------------------
// The gather kernel above issues one 4-byte load, one conversion and one select per K index and lane: 147 of each for a
// 7x7x3 filter, and the vector ALU, not memory, sets its time.  Here K is laid out as 21 (6x6: 18) (channel, filter row) pairs of
// 8 values each (7 taps + one zero): the 7 taps of a pair are 7 consecutive floats of one image row, so a lane fetches
// its half of a 16-wide K chunk with two 16-byte loads and converts it in place.  11 chunks (K = 176; 6x6: 9, K = 144) instead
// of 10, but a fifth of the instructions.  Loads go through a buffer resource: a vector that starts
// left of the image or ends past the tensor reads zeros or a neighbouring row, and whatever lies outside the image is
// blanked before the conversion (only in groups that touch the border), what is no tap -- the values behind the filter row, the 22nd pair of
// a 7x7 filter -- always: its weights are zero, but zero times an infinite pixel is not.
// 16-byte load through a buffer resource: the hardware checks the byte offset against the resource size and returns zeros
// beyond it (an index that went negative wraps to an offset past the end)
typedef int stemI32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t stemRsrc(const void *base, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ f32x4 stemLoad16(__amdgpu_buffer_rsrc_t r, unsigned voffset)
{
    const stemI32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(voffset), 0, 0);
    return __builtin_bit_cast(f32x4, v);
}

constexpr int stemRowChunks(int ks) { return (3 * ks + 1) / 2; }       // chunks of two (channel, filter row) pairs
constexpr int kRowChunksMost = stemRowChunks(7);

struct StemRowsArgs
{
    const float *x;
    const f16   *wA;        // [mBlocks][stemRowChunks(KS)][64 lanes][8]
    const float *scale;
    const float *shift;
    f16         *y;
    int B, H, W, OH, OW, outLd, outC, stride, pad;
    int groupsPerRow, nGroups;
    unsigned xBytes;
    int act;
    float actParam, outMul;
    int rowOff[2 * kRowChunksMost]; // (ci * H + ky) * W of pair r; padding pair: 0
    int rowKy[2 * kRowChunksMost];  // ky of pair r; padding pair: 32767 (never inside the image)
};

template <int KS, int MBLK>
__global__ __launch_bounds__(256) void convStemRowsKernel(StemRowsArgs a)
{
    touchArgs(a);
    constexpr int kRowChunks = stemRowChunks(KS);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    f16 *wl = reinterpret_cast<f16 *>(smem);                                        // [MBLK][kRowChunks][64][8]
    float *ssl = reinterpret_cast<float *>(smem + MBLK * kRowChunks * 1024);         // [2][MBLK*32]
    for (int i = threadIdx.x; i < MBLK * kRowChunks * 64; i += 256)
        reinterpret_cast<f16x8 *>(wl)[i] = reinterpret_cast<const f16x8 *>(a.wA)[i];
    for (int i = threadIdx.x; i < MBLK * 32; i += 256)
    {
        ssl[i] = a.scale && i < a.outC ? a.scale[i] : 1.f;
        ssl[MBLK * 32 + i] = a.shift && i < a.outC ? a.shift[i] : 0.f;
    }
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int n = lane & 31;
    const bool hi = lane >= 32;
    // (contiguous runs of pixel groups per workgroup, XCD by XCD: see convStemMfmaKernel)
    const int nBlocks = static_cast<int>(gridDim.x);
    const int perXcd = (nBlocks + 7) / 8;
    const int logical = static_cast<int>(blockIdx.x % 8) * perXcd + static_cast<int>(blockIdx.x / 8);
    const int perBlock = (a.nGroups + nBlocks - 1) / nBlocks;
    const int gBegin = logical < nBlocks ? logical * perBlock : a.nGroups;
    const int gEnd = min(a.nGroups, gBegin + perBlock);
    const int planes = 3 * a.H * a.W;
    const __amdgpu_buffer_rsrc_t rx = stemRsrc(a.x, a.xBytes);

    const bool lin = (a.act == MSNH_ACT_LEAKY || a.act == MSNH_ACT_RELU || a.act == MSNH_ACT_NONE);
    const float slope = a.act == MSNH_ACT_LEAKY ? a.actParam : (a.act == MSNH_ACT_RELU ? 0.f : 1.f);

    for (int g = gBegin + static_cast<int>(threadIdx.x >> 6); g < gEnd; g += 4)
    {
        const int gx = g % a.groupsPerRow;
        const int row = g / a.groupsPerRow;
        const int oy = row % a.OH;
        const int b = row / a.OH;
        const int ox = gx * 32 + n;
        const int iy0 = oy * a.stride - a.pad;
        const int ix0 = ox * a.stride - a.pad;
        const int base = b * planes + iy0 * a.W + ix0;             // element index of the window's corner; may be negative
        f32x16 acc[MBLK];
#pragma unroll
        for (int mb = 0; mb < MBLK; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;

        // wave-uniform: every tap of every pixel of the group lies inside the image (no blanking then)
        const int ixFirst = gx * 32 * a.stride - a.pad;
        const int ixLast  = (gx * 32 + 31) * a.stride - a.pad;
        const bool interior = iy0 >= 0 && iy0 + KS <= a.H && ixFirst >= 0 && ixLast + KS <= a.W && gx * 32 + 31 < a.OW;
        staticFor<0, kRowChunks>([&](auto cTag) {
            constexpr int c = decltype(cTag)::value;
            const int off = base + (hi ? a.rowOff[2 * c + 1] : a.rowOff[2 * c]);
            // a negative index wraps past the end of the buffer: zeros; so does the padding pair's
            const unsigned voff = 2 * c + 1 >= 3 * KS && hi ? 0x80000000u : static_cast<unsigned>(off) * 4u;
            f32x4 lo4 = stemLoad16(rx, voff);
            f32x4 hi4 = stemLoad16(rx, voff + 16u);
            float v[8] = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], KS > 6 ? hi4[2] : 0.f, 0.f};
            if (!interior)
            {
                const int ky = hi ? a.rowKy[2 * c + 1] : a.rowKy[2 * c];
                const bool rowOk = static_cast<unsigned>(iy0 + ky) < static_cast<unsigned>(a.H);
                if (off < 0 && rowOk)
                {
                    // the first image row of the first plane, left border: the 16-byte vectors would start in front of the
                    // tensor (and their offsets wrap), so the taps that exist are fetched one by one
#pragma unroll
                    for (int e = 0; e < KS; ++e)
                        v[e] = off + e >= 0 ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, (off + e) * 4, 0, 0)) : 0.f;
                }
#pragma unroll
                for (int e = 0; e < KS; ++e) v[e] = (rowOk && static_cast<unsigned>(ix0 + e) < static_cast<unsigned>(a.W)) ? v[e] : 0.f;
            }
            f16x8 bf;
#pragma unroll
            for (int e = 0; e < 8; ++e) bf[e] = static_cast<f16>(v[e]);
#pragma unroll
            for (int mb = 0; mb < MBLK; ++mb)
            {
                const f16x8 wa = *reinterpret_cast<const f16x8 *>(wl + ((static_cast<size_t>(mb) * kRowChunks + c) * 64 + lane) * 8);
                acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wa, bf, acc[mb], 0, 0, 0);
            }
        });
        if (ox < a.OW && (!hi || a.outC > 16))
        {
            f16 *yp = a.y + (static_cast<size_t>(row) * a.OW + ox) * a.outLd + (hi ? 16 : 0);
#pragma unroll
            for (int mb = 0; mb < MBLK; ++mb)
            {
                const float *scp = ssl + mb * 32 + (hi ? 16 : 0);
                const float *shp = scp + MBLK * 32;
                f16x8 o0, o1;
                float t[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) t[r] = acc[mb][r] * scp[r] + shp[r];
                if (lin)
                {
#pragma unroll
                    for (int r = 0; r < 16; ++r) t[r] = t[r] > 0.f ? t[r] : slope * t[r];
                }
                else activateArray<16>(t, a.act, a.actParam);
#pragma unroll
                for (int r = 0; r < 16; ++r)
                {
                    const float u = t[r] * a.outMul;
                    if (r < 8) o0[r] = static_cast<f16>(u); else o1[r - 8] = static_cast<f16>(u);
                }
                *reinterpret_cast<f16x8 *>(yp + mb * 32) = o0;
                *reinterpret_cast<f16x8 *>(yp + mb * 32 + 8) = o1;
            }
        }
    }
}

template <int KS, int MBLK>
int launchStemRows(const StemRowsArgs &a, unsigned blocks, hipStream_t st)
{
    const size_t smem = static_cast<size_t>(MBLK) * stemRowChunks(KS) * 1024 + 2 * MBLK * 32 * sizeof(float);
    auto kern = convStemRowsKernel<KS, MBLK>;
    if (const int rc = allowLds(reinterpret_cast<const void *>(kern), smem)) return rc;
    hipLaunchKernelGGL(kern, dim3((blocks + 7) / 8 * 8), dim3(256), smem, st, a);      // a multiple of 8: the XCD regrouping is a bijection then
    MSNH_LAUNCH_CHECK();
    return 0;
}

// the row-ordered kernel takes 7x7 and 6x6 filters over 3 channels whose whole input is addressable with 32-bit byte offsets
inline bool stemRowsOk(const msnh_conv_desc *d)
{
    return (d->ksize == 7 || d->ksize == 6) && d->in_c == 3 && static_cast<long long>(d->batch) * 3 * d->in_h * d->in_w * 4 < 0x7fffffffLL;
}

// ---- float32 networks ---------------------------------------------------------------------------------------------------------------
// 32x32x2 float32 MFMAs (a lane of the upper half holds the odd K index of a step), 64 clocks per step, block and SIMD: 7x7x3 -> 64 channels of one
// 224 x 224 image are 1.5 us of matrix-core time.  K is laid out by image rows as above: a step multiplies tap e of two (channel, filter row) pairs, the
// lower half of the wavefront holding the first pair's value and the upper half the second's, so a lane fetches the taps of its row with one or two
// 16-byte loads.  (The scalar kernel before it: one LDS broadcast and one FMA per filter value, 22.5 us for that image; K in tap order with a
// gather per value on the same MFMAs: 17.2; this one: 7.9, five images 54.8 -> 22.8.)  A small image is split over the channel blocks too (grid y), so that every SIMD has a wavefront.
struct StemF32Args
{
    const float *x;
    const float *wA;        // [mBlocks][ceil(steps / 4)][64 lanes][4]: four K steps per 16 bytes
    const float *scale;
    const float *shift;
    float       *y;
    int H, W, OH, OW, outLd, outC, stride, pad;
    int groupsPerRow, nGroups;
    int act;
    float actParam, outMul;
};

constexpr int stemF32Steps(int ks, int cin) { return (cin * ks + 1) / 2 * ks; }

template <int KS, int CIN, int MBLK>
__global__ __launch_bounds__(256) void convStemMfmaF32Kernel(StemF32Args a)
{
    touchArgs(a);
    constexpr int ROWS = CIN * KS, CHUNKS = (ROWS + 1) / 2, QUADS = (stemF32Steps(KS, CIN) + 3) / 4;
    constexpr int GC = 4;                                                          // chunks per group; 4 KS steps are whole quads
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    f32x4 *wl = reinterpret_cast<f32x4 *>(smem);                                  // [MBLK][QUADS][64]
    float *ssl = reinterpret_cast<float *>(smem + MBLK * QUADS * 1024);            // [2][MBLK*32]
    const int c0 = static_cast<int>(blockIdx.y) * MBLK * 32;
    for (int i = threadIdx.x; i < MBLK * QUADS * 64; i += 256) wl[i] = reinterpret_cast<const f32x4 *>(a.wA)[static_cast<size_t>(blockIdx.y) * MBLK * QUADS * 64 + i];
    for (int i = threadIdx.x; i < MBLK * 32; i += 256)
    {
        ssl[i] = a.scale && c0 + i < a.outC ? a.scale[c0 + i] : 1.f;
        ssl[MBLK * 32 + i] = a.shift && c0 + i < a.outC ? a.shift[c0 + i] : 0.f;
    }
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int n = lane & 31;
    const bool hi = lane >= 32;
    const int nBlocks = static_cast<int>(gridDim.x);
    const int perXcd = (nBlocks + 7) / 8;
    const int logical = static_cast<int>(blockIdx.x % 8) * perXcd + static_cast<int>(blockIdx.x / 8);     // (see convStemMfmaKernel)
    const int perBlock = (a.nGroups + nBlocks - 1) / nBlocks;
    const int gBegin = logical < nBlocks ? logical * perBlock : a.nGroups;
    const int gEnd = min(a.nGroups, gBegin + perBlock);
    const int planes = CIN * a.H * a.W;
    const bool lin = (a.act == MSNH_ACT_LEAKY || a.act == MSNH_ACT_RELU || a.act == MSNH_ACT_NONE);
    const float slope = a.act == MSNH_ACT_LEAKY ? a.actParam : (a.act == MSNH_ACT_RELU ? 0.f : 1.f);

    for (int g = gBegin + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)); g < gEnd; g += 4)
    {
        const int gx = g % a.groupsPerRow;
        const int row = g / a.groupsPerRow;
        const int oy = row % a.OH;
        const int b = row / a.OH;
        const int ox = gx * 32 + n;
        const int iy0 = oy * a.stride - a.pad;
        const int ix0 = ox * a.stride - a.pad;
        const __amdgpu_buffer_rsrc_t rx = stemRsrc(a.x + static_cast<size_t>(b) * planes, static_cast<unsigned>(planes) * 4u);
        const int base = iy0 * a.W + ix0;                          // element index of the window's corner in the image; may be negative
        f32x16 acc[MBLK];
#pragma unroll
        for (int mb = 0; mb < MBLK; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;
        const int ixFirst = gx * 32 * a.stride - a.pad;
        const int ixLast  = (gx * 32 + 31) * a.stride - a.pad;
        const bool interior = iy0 >= 0 && iy0 + KS <= a.H && ixFirst >= 0 && ixLast + KS <= a.W && gx * 32 + 31 < a.OW;
        // the rows' values are fetched a group of chunks ahead of the MFMAs that use them (all at once they would take the registers of a second wavefront)
        float v[2][GC][KS];
        const auto fetch = [&](auto gTag) {
            constexpr int g0 = decltype(gTag)::value;
            staticFor<g0 * GC, (g0 + 1) * GC < CHUNKS ? (g0 + 1) * GC : CHUNKS>([&](auto cTag) {
                constexpr int c = decltype(cTag)::value;
                constexpr int r0 = 2 * c, r1 = 2 * c + 1 < ROWS ? 2 * c + 1 : 2 * c;
                float (&t)[KS] = v[g0 % 2][c - g0 * GC];
                const int off = base + (hi ? (r1 / KS * a.H + r1 % KS) * a.W : (r0 / KS * a.H + r0 % KS) * a.W);
                // a negative index wraps past the end of the buffer: zeros; so does the padding pair's (zero filter values alone would not do: zero times
                // an infinite pixel is not zero)
                const bool padded = 2 * c + 1 >= ROWS && hi;
                const unsigned voff = padded ? 0x80000000u : static_cast<unsigned>(off) * 4u;
                const f32x4 lo4 = stemLoad16(rx, voff);
                f32x4 hi4 = {0.f, 0.f, 0.f, 0.f};
                if constexpr (KS > 5) hi4 = stemLoad16(rx, voff + 16u);
                else if constexpr (KS > 4) hi4[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, static_cast<int>(voff + 16u), 0, 0));
#pragma unroll
                for (int e = 0; e < KS; ++e) t[e] = e < 4 ? lo4[e & 3] : hi4[e & 3];
                if (!interior)
                {
                    const bool rowOk = !padded && static_cast<unsigned>(iy0 + (hi ? r1 % KS : r0 % KS)) < static_cast<unsigned>(a.H);
                    if (off < 0 && rowOk)
                    {
                        // the first image row of the first plane, left border: the 16-byte vectors would start in front of the tensor
#pragma unroll
                        for (int e = 0; e < KS; ++e)
                            t[e] = off + e >= 0 ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, (off + e) * 4, 0, 0)) : 0.f;
                    }
#pragma unroll
                    for (int e = 0; e < KS; ++e) t[e] = (rowOk && static_cast<unsigned>(ix0 + e) < static_cast<unsigned>(a.W)) ? t[e] : 0.f;
                }
            });
        };
        fetch(std::integral_constant<int, 0>());
        staticFor<0, (CHUNKS + GC - 1) / GC>([&](auto gTag) {
            constexpr int g0 = decltype(gTag)::value;
            if constexpr ((g0 + 1) * GC < CHUNKS) fetch(std::integral_constant<int, g0 + 1>());
            __builtin_amdgcn_sched_barrier(0);
            staticFor<g0 * GC * KS / 4, ((g0 + 1) * GC < CHUNKS ? (g0 + 1) * GC * KS / 4 : QUADS)>([&](auto qTag) {
                constexpr int q = decltype(qTag)::value;
#pragma unroll
                for (int mb = 0; mb < MBLK; ++mb)
                {
                    const f32x4 w4 = wl[(mb * QUADS + q) * 64 + lane];
                    staticFor<0, 4>([&](auto eTag) {
                        constexpr int s = 4 * q + decltype(eTag)::value;
                        if constexpr (s < CHUNKS * KS) acc[mb] = __builtin_amdgcn_mfma_f32_32x32x2f32(w4[s % 4], v[g0 % 2][s / KS - g0 * GC][s % KS], acc[mb], 0, 0, 0);
                    });
                }
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        if (ox < a.OW && (!hi || a.outC > 16))
        {
            float *yp = a.y + (static_cast<size_t>(row) * a.OW + ox) * a.outLd + c0 + (hi ? 16 : 0);
#pragma unroll
            for (int mb = 0; mb < MBLK; ++mb)
            {
                const float *scp = ssl + mb * 32 + (hi ? 16 : 0);
                const float *shp = scp + MBLK * 32;
                float t[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) t[r] = acc[mb][r] * scp[r] + shp[r];
                if (lin)
                {
#pragma unroll
                    for (int r = 0; r < 16; ++r) t[r] = t[r] > 0.f ? t[r] : slope * t[r];
                }
                else activateArray<16>(t, a.act, a.actParam);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f32x4 *>(yp + mb * 32 + 4 * q) = f32x4{t[4 * q] * a.outMul, t[4 * q + 1] * a.outMul, t[4 * q + 2] * a.outMul, t[4 * q + 3] * a.outMul};
            }
        }
    }
}

template <int KS, int CIN, int MBLK>
int launchStemF32(const StemF32Args &a, unsigned blocks, hipStream_t st)
{
    const size_t smem = static_cast<size_t>(MBLK) * ((stemF32Steps(KS, CIN) + 3) / 4) * 1024 + 2 * MBLK * 32 * sizeof(float);
    auto kern = convStemMfmaF32Kernel<KS, CIN, MBLK>;
    if (const int rc = allowLds(reinterpret_cast<const void *>(kern), smem)) return rc;
    hipLaunchKernelGGL(kern, dim3((blocks + 7) / 8 * 8, static_cast<unsigned>((a.outC + 31) / (32 * MBLK))), dim3(256), smem, st, a);
    MSNH_LAUNCH_CHECK();
    return 0;
}

// where K index k = tap * Cin + ci lies: offset inside one image's planes, and its filter row and column
inline void stemTaps(const msnh_conv_desc *d, int *koff, int *kyx)
{
    const int K = d->ksize * d->ksize * d->in_c;
    for (int k = 0; k < kStemMaxK; ++k)
    {
        const int tap = k / d->in_c, ci = k % d->in_c;
        const int ky = tap / d->ksize, kx = tap % d->ksize;
        koff[k] = k < K ? (ci * d->in_h + ky) * d->in_w + kx : 0;
        kyx[k] = k < K ? ky << 8 | kx : 32767 << 8;
    }
}

inline int stemMBlocks(const msnh_conv_desc *d) { return (d->out_c + 31) / 32; }
inline int stemKBlocks(const msnh_conv_desc *d) { return (d->ksize * d->ksize * d->in_c + 31) / 32; }

} // namespace

static bool stemMfmaShape(const msnh_conv_desc *d)
{
    const int mb = d->out_c / 32;              // (16 channels: half a block, the other half of its rows zero)
    return d->dtype == MSNH_F16 && d->out_dtype == MSNH_F16 && d->in_c >= 1 && d->in_c <= 4 &&
           d->ksize * d->ksize * d->in_c <= kStemMaxK && d->groups == 1 && d->dilation == 1 && (d->out_c == 16 || (d->out_c % 32 == 0 && (mb == 1 || mb == 2 || mb == 4))) &&
           d->out_ld % 8 == 0 && !d->has_residual && d->in_h < 30000;
}

static bool stemMfmaF32Shape(const msnh_conv_desc *d)
{
    return d->dtype == MSNH_F32 && d->out_dtype == MSNH_F32 && d->in_c >= 1 && d->in_c <= 4 &&
           d->ksize * d->ksize * d->in_c <= kStemMaxK && d->groups == 1 && d->dilation == 1 && (d->out_c == 16 || d->out_c % 32 == 0) && d->out_ld % 4 == 0 && !d->has_residual &&
           d->in_h < 30000 && static_cast<long long>(d->in_c) * d->in_h * d->in_w * 4 < 0x7fffffffLL;
}

static bool stemSize(const msnh_conv_desc *d) { return d->ksize == 3 || d->ksize == 5 || d->ksize == 7; }

bool stemMfmaOk(const msnh_conv_desc *d) { return stemSize(d) && stemMfmaShape(d); }
bool stemMfmaF32Ok(const msnh_conv_desc *d) { return stemSize(d) && stemMfmaF32Shape(d); }
bool stemFocusOk(const msnh_conv_desc *d)
{
    return d->ksize == 6 && d->stride == 2 && d->pad == 2 && d->in_c <= 3 && (stemMfmaShape(d) || stemMfmaF32Shape(d));
}

size_t stemMfmaF32Elems(const msnh_conv_desc *d) { return static_cast<size_t>(stemMBlocks(d)) * ((stemF32Steps(d->ksize, d->in_c) + 3) / 4) * 256; }

// packed[mb][step / 4][lane][step % 4] = W[channel(mb, lane % 32)][ci][ky][kx], kx = step % ksize, (ci, ky) = pair 2 * (step / ksize) + lane / 32
void stemMfmaF32Pack(const msnh_conv_desc *d, const float *oihw, float *packed)
{
    const int ks = d->ksize, steps = stemF32Steps(ks, d->in_c), quads = (steps + 3) / 4;
    for (int mb = 0; mb < stemMBlocks(d); ++mb)
        for (int s = 0; s < quads * 4; ++s)
            for (int lane = 0; lane < 64; ++lane)
            {
                const int m = lane % 32;
                const int oc = mb * 32 + 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
                const int pair = 2 * (s / ks) + lane / 32;
                const bool real = s < steps && pair < d->in_c * ks && oc < d->out_c;
                packed[(static_cast<size_t>(mb * quads + s / 4) * 64 + lane) * 4 + s % 4] =
                    real ? oihw[((static_cast<size_t>(oc) * d->in_c + pair / ks) * ks + pair % ks) * ks + s % ks] : 0.f;
            }
}

size_t stemMfmaElems(const msnh_conv_desc *d)
{
    return static_cast<size_t>(stemMBlocks(d)) * (stemRowsOk(d) ? stemRowChunks(d->ksize) : stemKBlocks(d) * 2) * 64 * 8;
}

// packed[mb][kb16][lane][e] = W[channel(mb, lane % 32)][k = kb16*16 + 8*(lane/32) + e], k = tap*Cin + ci
void stemMfmaPack(const msnh_conv_desc *d, const float *oihw, _Float16 *packed)
{
    const int cin = d->in_c, kk = d->ksize * d->ksize, K = kk * cin, KB2 = stemKBlocks(d) * 2;
    if (stemRowsOk(d))
    {
        // packed[mb][chunk][lane][e] = W[channel(mb, lane % 32)][ci][ky][kx = e], (ci, ky) = pair 2 * chunk + lane / 32
        const int ks = d->ksize, chunks = stemRowChunks(ks);
        for (int mb = 0; mb < stemMBlocks(d); ++mb)
            for (int c = 0; c < chunks; ++c)
                for (int lane = 0; lane < 64; ++lane)
                    for (int e = 0; e < 8; ++e)
                    {
                        const int m = lane % 32;
                        const int oc = mb * 32 + 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
                        const int pair = 2 * c + lane / 32;
                        float v = 0.f;
                        if (pair < 3 * ks && e < ks && oc < d->out_c) v = oihw[((static_cast<size_t>(oc) * 3 + pair / ks) * ks + pair % ks) * ks + e];
                        packed[((static_cast<size_t>(mb) * chunks + c) * 64 + lane) * 8 + e] = static_cast<_Float16>(v);
                    }
        return;
    }
    for (int mb = 0; mb < stemMBlocks(d); ++mb)
        for (int kb = 0; kb < KB2; ++kb)
            for (int lane = 0; lane < 64; ++lane)
                for (int e = 0; e < 8; ++e)
                {
                    const int m = lane % 32;
                    const int oc = mb * 32 + 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
                    const int k = kb * 16 + 8 * (lane / 32) + e;
                    float v = 0.f;
                    if (k < K && oc < d->out_c)
                    {
                        const int tap = k / cin, ci = k % cin;
                        v = oihw[(static_cast<size_t>(oc) * cin + ci) * kk + tap];
                    }
                    packed[((static_cast<size_t>(mb) * KB2 + kb) * 64 + lane) * 8 + e] = static_cast<_Float16>(v);
                }
}

int convStemMfma(const msnh_conv_desc *d, const float *x, const _Float16 *wA, const float *scale, const float *shift, void *y, hipStream_t st)
{
    MSNH_REQUIRE(stemMfmaOk(d) || (stemFocusOk(d) && d->dtype == MSNH_F16), "conv2d: shape not supported by the matrix-core stem kernel");
    MSNH_REQUIRE(reinterpret_cast<uintptr_t>(y) % 16 == 0 && reinterpret_cast<uintptr_t>(wA) % 16 == 0, "conv2d: stem needs 16-byte aligned output and weights");
    if (stemRowsOk(d))
    {
        StemRowsArgs r;
        r.x = x; r.wA = wA; r.scale = scale; r.shift = shift; r.y = static_cast<f16 *>(y);
        r.B = d->batch; r.H = d->in_h; r.W = d->in_w; r.OH = d->out_h; r.OW = d->out_w; r.outLd = d->out_ld; r.stride = d->stride; r.pad = d->pad;
        r.groupsPerRow = (d->out_w + 31) / 32;
        const long long groups = static_cast<long long>(d->batch) * d->out_h * r.groupsPerRow;
        MSNH_REQUIRE(groups < (1LL << 31), "conv2d: stem tensor too large");
        r.nGroups = static_cast<int>(groups);
        r.xBytes = static_cast<unsigned>(static_cast<long long>(d->batch) * 3 * d->in_h * d->in_w * 4);
        r.outC = d->out_c; r.act = d->act; r.actParam = d->act_param; r.outMul = d->out_mul;
        const int ks = d->ksize;
        for (int p = 0; p < 2 * kRowChunksMost; ++p)
        {
            r.rowOff[p] = p < 3 * ks ? ((p / ks) * d->in_h + p % ks) * d->in_w : 0;
            r.rowKy[p] = p < 3 * ks ? p % ks : 32767;
        }
        const long long want = (groups + 3) / 4;
        const unsigned blocks = static_cast<unsigned>(want < 256 * 4 ? (want < 1 ? 1 : want) : 256 * 4);     // (2..8 workgroups per CU measure alike)
        switch (stemMBlocks(d))
        {
        case 1: return ks == 6 ? launchStemRows<6, 1>(r, blocks, st) : launchStemRows<7, 1>(r, blocks, st);
        case 2: return ks == 6 ? launchStemRows<6, 2>(r, blocks, st) : launchStemRows<7, 2>(r, blocks, st);
        default: return ks == 6 ? launchStemRows<6, 4>(r, blocks, st) : launchStemRows<7, 4>(r, blocks, st);
        }
    }
    StemArgs a;
    a.x = x; a.wA = wA; a.scale = scale; a.shift = shift; a.y = static_cast<f16 *>(y);
    a.B = d->batch; a.H = d->in_h; a.W = d->in_w; a.OH = d->out_h; a.OW = d->out_w; a.outLd = d->out_ld; a.outC = d->out_c;
    a.stride = d->stride; a.pad = d->pad; a.cin = d->in_c; a.ksize = d->ksize;
    a.groupsPerRow = (d->out_w + 31) / 32;
    const long long groups = static_cast<long long>(d->batch) * d->out_h * a.groupsPerRow;
    MSNH_REQUIRE(groups < (1LL << 31) && static_cast<long long>(d->in_c) * d->in_h * d->in_w < (1LL << 31), "conv2d: stem tensor too large");
    a.nGroups = static_cast<int>(groups);
    a.act = d->act; a.actParam = d->act_param; a.outMul = d->out_mul;
    stemTaps(d, a.koff, a.kyx);
    // several wavefronts per SIMD hide the gather latency; every wavefront walks the pixel groups with a grid stride
    const long long want = (groups + 3) / 4;
    const int taps = d->ksize * d->ksize * d->in_c, mb = stemMBlocks(d);
    const long long cap = 256 * (taps <= 64 ? 8 : 4);             // measured: short K wants more wavefronts in flight
    const unsigned blocks = static_cast<unsigned>(want < cap ? (want < 1 ? 1 : want) : cap);
#define MSNH_STEM(T) if (taps == T) return mb <= 1 ? launchStem<T, 1>(a, blocks, st) : mb == 2 ? launchStem<T, 2>(a, blocks, st) : launchStem<T, 4>(a, blocks, st)
    MSNH_STEM(9); MSNH_STEM(18); MSNH_STEM(27); MSNH_STEM(36);                  // 3x3 over 1 to 4 channels
    MSNH_STEM(25); MSNH_STEM(50); MSNH_STEM(75); MSNH_STEM(100);                // 5x5
    MSNH_STEM(72); MSNH_STEM(108);                                              // 6x6 (over one channel: 36, above; over 3 a tensor too large for the row-ordered kernel)
    MSNH_STEM(49); MSNH_STEM(98); MSNH_STEM(147);                               // 7x7 (over 3 channels a tensor too large for the row-ordered kernel)
#undef MSNH_STEM
    setError("conv2d: stem shape not instantiated");
    return 2;
}

int convStemMfmaF32(const msnh_conv_desc *d, const float *x, const float *wA, const float *scale, const float *shift, float *y, hipStream_t st)
{
    MSNH_REQUIRE(stemMfmaF32Ok(d) || (stemFocusOk(d) && d->dtype == MSNH_F32), "conv2d: shape not supported by the matrix-core stem kernel");
    MSNH_REQUIRE(reinterpret_cast<uintptr_t>(y) % 16 == 0 && reinterpret_cast<uintptr_t>(wA) % 16 == 0, "conv2d: stem needs 16-byte aligned output and weights");
    StemF32Args a;
    a.x = x; a.wA = wA; a.scale = scale; a.shift = shift; a.y = y;
    a.H = d->in_h; a.W = d->in_w; a.OH = d->out_h; a.OW = d->out_w; a.outLd = d->out_ld; a.outC = d->out_c;
    a.stride = d->stride; a.pad = d->pad;
    a.groupsPerRow = (d->out_w + 31) / 32;
    const long long groups = static_cast<long long>(d->batch) * d->out_h * a.groupsPerRow;
    MSNH_REQUIRE(groups < (1LL << 31), "conv2d: stem tensor too large");
    a.nGroups = static_cast<int>(groups);
    a.act = d->act; a.actParam = d->act_param; a.outMul = d->out_mul;
    const long long want = (groups + 3) / 4;
    const unsigned blocks = static_cast<unsigned>(want < 256 * 4 ? (want < 1 ? 1 : want) : 256 * 4);
    // two channel blocks per wavefront share a gather where that still leaves two wavefronts per SIMD
    const int ks = d->ksize, cin = d->in_c, mb = d->out_c % 64 == 0 && groups * (d->out_c / 64) >= 2048 ? 2 : 1;
#define MSNH_STEM(KSV, CV) if (ks == KSV && cin == CV) return mb == 2 ? launchStemF32<KSV, CV, 2>(a, blocks, st) : launchStemF32<KSV, CV, 1>(a, blocks, st)
    MSNH_STEM(3, 1); MSNH_STEM(3, 2); MSNH_STEM(3, 3); MSNH_STEM(3, 4);
    MSNH_STEM(5, 1); MSNH_STEM(5, 2); MSNH_STEM(5, 3); MSNH_STEM(5, 4);
    MSNH_STEM(6, 1); MSNH_STEM(6, 2); MSNH_STEM(6, 3);
    MSNH_STEM(7, 1); MSNH_STEM(7, 2); MSNH_STEM(7, 3);
#undef MSNH_STEM
    setError("conv2d: stem shape not instantiated");
    return 2;
}

} // namespace msnh
