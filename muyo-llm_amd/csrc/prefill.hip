// Batched-prefill kernels for gfx950: the row-wise glue (embedding, rms_norm into split planes,
// rope + cache append) and the entry points of all of them. The GEMMs are in prefill_gemm.hip, the
// attention in prefill_attention.hip.
#include <algorithm>
#include <cmath>
#include <initializer_list>
#include <type_traits>

#include "prefill.hpp"
#include "prefill_core.hpp"

namespace muyo
{
namespace
{
// ------------------------------------------------------------------------------------------------
// Row-wise glue.

__global__ __launch_bounds__(256) void EmbedRowsKernel(const uint16_t* __restrict__ table,
                                                       const int32_t* __restrict__ tokens, uint32_t hidden,
                                                       float* __restrict__ x, int32_t* history, int32_t pos0,
                                                       uint32_t historyCap)
{
    const uint32_t m = blockIdx.x;
    const int32_t token = tokens[m];
    const uint16_t* row = table + static_cast<uint64_t>(token) * hidden;
    float* out = x + static_cast<uint64_t>(m) * hidden;
    for (uint32_t i = threadIdx.x; i < hidden; i += 256)
    {
        out[i] = HalfBitsToFloat(row[i]);
    }
    const int64_t position = static_cast<int64_t>(pos0) + m;
    if (threadIdx.x == 0 && history != nullptr && position >= 0 && position < historyCap)
    {
        history[position] = token;
    }
}

/// The K splits of a split GEMM folded into its consumer: x = residual + (P_0 + P_1 + ...) in
/// split order, the unsplit epilogue's residual + sum.
struct SplitSum
{
    const float* residual;  // may be null
    const float* partial;   // [splits][rows][cols]
    uint32_t splits;
    uint64_t stride;        // rows * cols

    __device__ float4 At(uint64_t i) const
    {
        float4 a = *reinterpret_cast<const float4*>(partial + i);
        for (uint32_t z = 1; z < splits; ++z)
        {
            const float4 b = *reinterpret_cast<const float4*>(partial + z * stride + i);
            a.x += b.x;
            a.y += b.y;
            a.z += b.z;
            a.w += b.w;
        }
        if (residual != nullptr)
        {
            const float4 r = *reinterpret_cast<const float4*>(residual + i);
            a = make_float4(r.x + a.x, r.y + a.y, r.z + a.z, r.w + a.w);
        }
        return a;
    }
};

/// One wave per row: sum of squares across the wave, then (scale * x) * w split into planes. With
/// a split sum (splits > 0) the row is first reduced from its parts and stored to x; without w
/// only that.
__global__ __launch_bounds__(256) void RmsNormSplitKernel(float* __restrict__ x, const float* __restrict__ w,
                                                          uint32_t rows, uint32_t cols, float eps,
                                                          uint16_t* __restrict__ hi, uint16_t* __restrict__ lo,
                                                          SplitSum sum)
{
    const uint32_t row = blockIdx.x * 4 + threadIdx.x / kWave;
    if (row >= rows)
    {
        return;
    }
    const uint32_t lane = threadIdx.x % kWave;
    float* xr = x + static_cast<uint64_t>(row) * cols;
    float ss = 0.0f;
    for (uint32_t i = lane * 4; i < cols; i += 4 * kWave)
    {
        float4 v;
        if (sum.splits > 0)
        {
            v = sum.At(static_cast<uint64_t>(row) * cols + i);
            *reinterpret_cast<float4*>(xr + i) = v;  // read back below by this lane only
        }
        else
        {
            v = *reinterpret_cast<const float4*>(xr + i);
        }
        ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
    if (w == nullptr)
    {
        return;
    }
    ss = GroupSum<kWave>(ss);
    const float scale = 1.0f / sqrtf(ss / static_cast<float>(cols) + eps);
    for (uint32_t i = lane * 4; i < cols; i += 4 * kWave)
    {
        const float4 v = *reinterpret_cast<const float4*>(xr + i);
        const float4 g = *reinterpret_cast<const float4*>(w + i);
        StoreSplit4(hi, lo, static_cast<uint64_t>(row) * cols + i, (scale * v.x) * g.x, (scale * v.y) * g.y,
                    (scale * v.z) * g.z, (scale * v.w) * g.w);
    }
}

/// RmsNormSplitKernel with kT threads per row (one wave, or the whole 256-thread workgroup) and
/// at most kChunks 16-byte chunks of the row per thread (and kParts K splits), all requested before
/// the first is used: every K split's part, the residual and the weight in one round of loads
/// instead of one round per chunk. The sums run in SplitSum::At's order; the sum of squares meets across the row's
/// waves in LDS.
template <int kT, uint32_t kParts>
__global__ __launch_bounds__(256) void RmsNormSplitRowsKernel(float* __restrict__ x, const float* __restrict__ w,
                                                              uint32_t rows, uint32_t cols, float eps,
                                                              uint16_t* __restrict__ hi, uint16_t* __restrict__ lo,
                                                              SplitSum sum)
{
    constexpr int kChunks = 4;
    constexpr int kRowsPerBlock = 256 / kT;
    constexpr int kWavesPerRow = kT / kWave;
    __shared__ float squares[kRowsPerBlock * kWavesPerRow];
    const uint32_t row = blockIdx.x * kRowsPerBlock + threadIdx.x / kT;
    const uint32_t t = threadIdx.x % kT;
    const bool live = row < rows;
    const uint64_t base = static_cast<uint64_t>(live ? row : 0) * cols;
    float4 v[kChunks];
    float4 part[kParts - 1][kChunks];
    float4 res[kChunks];
    float4 g[kChunks];
#pragma unroll
    for (int c = 0; c < kChunks; ++c)
    {
        const uint32_t i = (t + c * kT) * 4;
        const bool in = i < cols;
        const uint64_t at = base + (in ? i : 0);
        v[c] = *reinterpret_cast<const float4*>((sum.splits > 0 ? sum.partial : x) + at);
#pragma unroll
        for (uint32_t z = 1; z < kParts; ++z)
        {
            if (z < sum.splits)
            {
                part[z - 1][c] = *reinterpret_cast<const float4*>(sum.partial + z * sum.stride + at);
            }
        }
        if (sum.splits > 0 && sum.residual != nullptr)
        {
            res[c] = *reinterpret_cast<const float4*>(sum.residual + at);
        }
        if (w != nullptr)
        {
            g[c] = *reinterpret_cast<const float4*>(w + (in ? i : 0));
        }
    }
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < kChunks; ++c)
    {
        const uint32_t i = (t + c * kT) * 4;
        if (sum.splits > 0)
        {
#pragma unroll
            for (uint32_t z = 1; z < kParts; ++z)
            {
                if (z < sum.splits)
                {
                    v[c].x += part[z - 1][c].x;
                    v[c].y += part[z - 1][c].y;
                    v[c].z += part[z - 1][c].z;
                    v[c].w += part[z - 1][c].w;
                }
            }
            if (sum.residual != nullptr)
            {
                v[c] = make_float4(res[c].x + v[c].x, res[c].y + v[c].y, res[c].z + v[c].z, res[c].w + v[c].w);
            }
            if (live && i < cols)
            {
                *reinterpret_cast<float4*>(x + base + i) = v[c];
            }
        }
        if (i < cols)
        {
            ss += v[c].x * v[c].x + v[c].y * v[c].y + v[c].z * v[c].z + v[c].w * v[c].w;
        }
    }
    if (w == nullptr)
    {
        return;
    }
    ss = GroupSum<kWave>(ss);
    if constexpr (kWavesPerRow > 1)
    {
        const uint32_t wave = threadIdx.x / kWave;
        if (threadIdx.x % kWave == 0)
        {
            squares[wave] = ss;
        }
        __syncthreads();
        const uint32_t first = (threadIdx.x / kT) * kWavesPerRow;
        ss = 0.0f;
#pragma unroll
        for (int k = 0; k < kWavesPerRow; ++k)
        {
            ss += squares[first + k];
        }
    }
    if (!live)
    {
        return;
    }
    const float scale = 1.0f / sqrtf(ss / static_cast<float>(cols) + eps);
#pragma unroll
    for (int c = 0; c < kChunks; ++c)
    {
        const uint32_t i = (t + c * kT) * 4;
        if (i < cols)
        {
            StoreSplit4(hi, lo, base + i, (scale * v[c].x) * g[c].x, (scale * v[c].y) * g[c].y,
                        (scale * v[c].z) * g[c].z, (scale * v[c].w) * g[c].w);
        }
    }
}

/// The row kernel for `cols`: a wave per row up to 1024 columns, the workgroup per row up to 4096,
/// else the loop kernel. Sums of up to four parts keep their own kernel: the registers that eight
/// parts take halve the waves in flight.
hipError_t LaunchRmsNormSplitRows(hipStream_t s, float* x, const float* w, uint32_t rows, uint32_t cols, float eps,
                                  uint16_t* hi, uint16_t* lo, const SplitSum& sum)
{
    static_assert(kMaxGemmSplits == 8, "parts");
    const bool few = sum.splits <= 4;
    if (cols <= 4 * 4 * kWave)
    {
        hipLaunchKernelGGL((few ? RmsNormSplitRowsKernel<kWave, 4> : RmsNormSplitRowsKernel<kWave, 8>),
                           dim3(CeilDiv(rows, 4)), dim3(256), 0, s, x, w, rows, cols, eps, hi, lo, sum);
    }
    else if (cols <= 4 * 4 * 256)
    {
        hipLaunchKernelGGL((few ? RmsNormSplitRowsKernel<256, 4> : RmsNormSplitRowsKernel<256, 8>), dim3(rows),
                           dim3(256), 0, s, x, w, rows, cols, eps, hi, lo, sum);
    }
    else
    {
        hipLaunchKernelGGL(RmsNormSplitKernel, dim3(CeilDiv(rows, 4)), dim3(256), 0, s, x, w, rows, cols, eps, hi, lo,
                           sum);
    }
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void SplitF32Kernel(const float* __restrict__ x, uint64_t quads,
                                                      uint16_t* __restrict__ hi, uint16_t* __restrict__ lo)
{
    for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < quads; i += static_cast<uint64_t>(gridDim.x) * 256)
    {
        const float4 v = *reinterpret_cast<const float4*>(x + 4 * i);
        StoreSplit4(hi, lo, 4 * i, v.x, v.y, v.z, v.w);
    }
}

/// The decode step's rope and cache append (rope_funcs.glsl:76-114; the fp16 cache rows of
/// src/FullModel.cpp:771-784) for many positions: one thread per (row, unit), units as in the
/// decode QKV epilogue: rope pairs (j, j + hd/2) of each q and k head, then pairs of v channels.
/// With splits > 1, qkv holds the K splits' raw sums ([splits][rows][width]) and each value is
/// their sum plus bias, the unsplit epilogue's acc + bias.
__global__ __launch_bounds__(256) void RopeSplitAppendKernel(const float* __restrict__ qkv, uint32_t rows,
                                                             int32_t pos0, uint32_t heads, uint32_t kvHeads,
                                                             uint32_t headDim, uint32_t maxSeq,
                                                             const float* __restrict__ ropePow,
                                                             uint16_t* __restrict__ qhi, uint16_t* __restrict__ qlo,
                                                             uint16_t* __restrict__ kcache,
                                                             uint16_t* __restrict__ vcache, uint32_t splits,
                                                             const float* __restrict__ bias)
{
    const uint32_t half = headDim / 2;
    const uint32_t ropeUnits = (heads + kvHeads) * half;
    const uint32_t units = (heads + 2 * kvHeads) * half;
    const uint64_t index = blockIdx.x * 256ull + threadIdx.x;
    if (index >= static_cast<uint64_t>(rows) * units)
    {
        return;
    }
    const uint32_t m = static_cast<uint32_t>(index / units);
    const uint32_t unit = static_cast<uint32_t>(index % units);
    const int32_t pos = pos0 + static_cast<int32_t>(m);
    const uint32_t width = (heads + 2 * kvHeads) * headDim;
    const float* row = qkv + static_cast<uint64_t>(m) * width;
    const uint64_t stride = static_cast<uint64_t>(rows) * width;
    auto value = [&](uint32_t col) {
        if (splits <= 1)
        {
            return row[col];
        }
        float a = row[col];
        for (uint32_t z = 1; z < splits; ++z)
        {
            a += row[z * stride + col];
        }
        return a + bias[col];
    };
    if (unit < ropeUnits)
    {
        const uint32_t head = unit / half;
        const uint32_t j = unit % half;
        const float s0 = value(head * headDim + j);
        const float s1 = value(head * headDim + j + half);
        const float theta = static_cast<float>(pos) * ropePow[j];
        float c;
        float sn;
        sincosf(theta, &sn, &c);
        const float o0 = s0 * c - s1 * sn;
        const float o1 = s0 * sn + s1 * c;
        if (head < heads)
        {
            const uint64_t at = static_cast<uint64_t>(m) * heads * headDim + head * headDim + j;
            const _Float16 h0 = HiHalf(o0);
            const _Float16 h1 = HiHalf(o1);
            qhi[at] = __builtin_bit_cast(uint16_t, h0);
            qlo[at] = __builtin_bit_cast(uint16_t, LoHalf(o0));
            qhi[at + half] = __builtin_bit_cast(uint16_t, h1);
            qlo[at + half] = __builtin_bit_cast(uint16_t, LoHalf(o1));
        }
        else
        {
            const uint64_t base = (static_cast<uint64_t>(head - heads) * maxSeq + pos) * headDim;
            kcache[base + j] = FloatToHalfBits(o0);
            kcache[base + j + half] = FloatToHalfBits(o1);
        }
    }
    else
    {
        const uint32_t channel = 2 * (unit - ropeUnits);  // within kvHeads * headDim
        const uint32_t g = channel / headDim;
        const uint64_t base = (static_cast<uint64_t>(g) * maxSeq + pos) * headDim + channel % headDim;
        const uint32_t v = (heads + kvHeads) * headDim + channel;
        vcache[base] = FloatToHalfBits(value(v));
        vcache[base + 1] = FloatToHalfBits(value(v + 1));
    }
}

/// RopeSplitAppendKernel with four pairs (or four v channels) per thread: 16-byte loads, 8-byte
/// stores and the same arithmetic per element (head_dim % 8 == 0, buffers aligned). The table of
/// powers is requested before the partial sums, so the angles are computed while the sums are
/// in flight (loads complete in order).
///
/// kParts is the most K splits summed, all requested before the first is added; 1 means whole sums
/// (bias included) in qkv. The parts' registers cost waves in flight: whole sums of 28 / 4 heads of
/// 128, 1024 rows, 7.0 us through the eight-part kernel (108 registers, four waves per SIMD), 6.2
/// through the one-part kernel (44, eight); 2048 rows 12.5 / 12.0.
template <uint32_t kParts>
__global__ __launch_bounds__(256) void RopeSplitAppendQuadKernel(const float* __restrict__ qkv, uint32_t rows,
                                                                 int32_t pos0, uint32_t heads, uint32_t kvHeads,
                                                                 uint32_t headDim, uint32_t maxSeq,
                                                                 const float* __restrict__ ropePow,
                                                                 uint16_t* __restrict__ qhi, uint16_t* __restrict__ qlo,
                                                                 uint16_t* __restrict__ kcache,
                                                                 uint16_t* __restrict__ vcache, uint32_t splits,
                                                                 const float* __restrict__ bias)
{
    const uint32_t half = headDim / 2;
    const uint32_t quads = half / 4;
    const uint32_t ropeUnits = (heads + kvHeads) * quads;
    const uint32_t units = ropeUnits + kvHeads * headDim / 4;
    const uint64_t index = blockIdx.x * 256ull + threadIdx.x;
    if (index >= static_cast<uint64_t>(rows) * units)
    {
        return;
    }
    const uint32_t m = static_cast<uint32_t>(index / units);
    const uint32_t unit = static_cast<uint32_t>(index % units);
    const int32_t pos = pos0 + static_cast<int32_t>(m);
    const uint32_t width = (heads + 2 * kvHeads) * headDim;
    const float* row = qkv + static_cast<uint64_t>(m) * width;
    const uint64_t stride = static_cast<uint64_t>(rows) * width;
    struct Parts
    {
        float4v v[kParts];
        float4v bias;
    };
    auto request = [&](uint32_t col) {
        Parts p;
        p.v[0] = *reinterpret_cast<const float4v*>(row + col);
        if constexpr (kParts > 1)
        {
#pragma unroll
            for (uint32_t z = 1; z < kParts; ++z)
            {
                if (z < splits)
                {
                    p.v[z] = *reinterpret_cast<const float4v*>(row + z * stride + col);
                }
            }
            p.bias = *reinterpret_cast<const float4v*>(bias + col);
        }
        return p;
    };
    auto total = [&](const Parts& p) {
        float4v a = p.v[0];
        if constexpr (kParts > 1)
        {
#pragma unroll
            for (uint32_t z = 1; z < kParts; ++z)
            {
                if (z < splits)
                {
                    a += p.v[z];
                }
            }
            a += p.bias;
        }
        return a;
    };
    if (unit < ropeUnits)
    {
        const uint32_t head = unit / quads;
        const uint32_t j = (unit % quads) * 4;
        const float4v power = *reinterpret_cast<const float4v*>(ropePow + j);
        const Parts p0 = request(head * headDim + j);
        const Parts p1 = request(head * headDim + j + half);
        float c[4];
        float sn[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            const float theta = static_cast<float>(pos) * power[e];
            sincosf(theta, &sn[e], &c[e]);
        }
        const float4v s0 = total(p0);
        const float4v s1 = total(p1);
        float o0[4];
        float o1[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            o0[e] = s0[e] * c[e] - s1[e] * sn[e];
            o1[e] = s0[e] * sn[e] + s1[e] * c[e];
        }
        if (head < heads)
        {
            const uint64_t at = static_cast<uint64_t>(m) * heads * headDim + head * headDim + j;
            StoreSplit4(qhi, qlo, at, o0[0], o0[1], o0[2], o0[3]);
            StoreSplit4(qhi, qlo, at + half, o1[0], o1[1], o1[2], o1[3]);
        }
        else
        {
            const uint64_t base = (static_cast<uint64_t>(head - heads) * maxSeq + pos) * headDim + j;
            const ushort4v k0 = {FloatToHalfBits(o0[0]), FloatToHalfBits(o0[1]), FloatToHalfBits(o0[2]),
                                 FloatToHalfBits(o0[3])};
            const ushort4v k1 = {FloatToHalfBits(o1[0]), FloatToHalfBits(o1[1]), FloatToHalfBits(o1[2]),
                                 FloatToHalfBits(o1[3])};
            *reinterpret_cast<ushort4v*>(kcache + base) = k0;
            *reinterpret_cast<ushort4v*>(kcache + base + half) = k1;
        }
    }
    else
    {
        const uint32_t channel = 4 * (unit - ropeUnits);  // within kvHeads * headDim
        const uint32_t g = channel / headDim;
        const uint64_t base = (static_cast<uint64_t>(g) * maxSeq + pos) * headDim + channel % headDim;
        const float4v v = total(request((heads + kvHeads) * headDim + channel));
        const ushort4v out = {FloatToHalfBits(v[0]), FloatToHalfBits(v[1]), FloatToHalfBits(v[2]),
                              FloatToHalfBits(v[3])};
        *reinterpret_cast<ushort4v*>(vcache + base) = out;
    }
}

}  // namespace

hipError_t LaunchEmbedRows(hipStream_t s, const uint16_t* table, const int32_t* tokens, uint32_t rows,
                           uint32_t hidden, float* x, int32_t* history, int32_t pos0, uint32_t historyCap)
{
    hipLaunchKernelGGL(EmbedRowsKernel, dim3(rows), dim3(256), 0, s, table, tokens, hidden, x, history, pos0,
                       historyCap);
    return hipGetLastError();
}

hipError_t LaunchRmsNormSplit(hipStream_t s, const float* x, const float* w, uint32_t rows, uint32_t cols, float eps,
                              uint16_t* hi, uint16_t* lo)
{
    if (rows == 0 || cols == 0 || cols % 4 != 0 || w == nullptr)
    {
        return hipErrorInvalidValue;
    }
    return LaunchRmsNormSplitRows(s, const_cast<float*>(x), w, rows, cols, eps, hi, lo, SplitSum{});
}

hipError_t LaunchReduceRmsNormSplit(hipStream_t s, const float* residual, const float* partial, uint32_t splits,
                                    float* x, const float* w, uint32_t rows, uint32_t cols, float eps, uint16_t* hi,
                                    uint16_t* lo)
{
    if (rows == 0 || cols == 0 || cols % 4 != 0 || splits == 0 || splits > kMaxGemmSplits || partial == nullptr)
    {
        return hipErrorInvalidValue;
    }
    const SplitSum sum{residual, partial, splits, static_cast<uint64_t>(rows) * cols};
    return LaunchRmsNormSplitRows(s, x, w, rows, cols, eps, hi, lo, sum);
}

hipError_t LaunchSplitF32(hipStream_t s, const float* x, uint64_t count, uint16_t* hi, uint16_t* lo)
{
    if (count == 0 || count % 4 != 0)
    {
        return hipErrorInvalidValue;
    }
    const uint64_t quads = count / 4;
    const uint32_t blocks = static_cast<uint32_t>(quads / 256 + 1 < 4096 ? quads / 256 + 1 : 4096);
    hipLaunchKernelGGL(SplitF32Kernel, dim3(blocks), dim3(256), 0, s, x, quads, hi, lo);
    return hipGetLastError();
}

hipError_t LaunchRopeSplitAppend(hipStream_t s, const float* qkv, uint32_t rows, int32_t pos0, uint32_t heads,
                                 uint32_t kvHeads, uint32_t headDim, uint32_t maxSeq, const float* ropePow,
                                 uint16_t* qhi, uint16_t* qlo, uint16_t* kcache, uint16_t* vcache, uint32_t splits,
                                 const float* bias)
{
    const uint64_t total = static_cast<uint64_t>(rows) * (heads + 2 * kvHeads) * (headDim / 2);
    if (total == 0 || pos0 < 0 || static_cast<uint64_t>(pos0) + rows > maxSeq || splits == 0 ||
        splits > kMaxGemmSplits || (splits > 1 && bias == nullptr))
    {
        return hipErrorInvalidValue;
    }
    const auto aligned = [](const void* p, uintptr_t bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; };
    if (headDim % 8 == 0 && aligned(qkv, 16) && aligned(ropePow, 16) && (bias == nullptr || aligned(bias, 16)) &&
        aligned(qhi, 8) && aligned(qlo, 8) && aligned(kcache, 8) && aligned(vcache, 8))
    {
        // Threads: four pairs of a rotated head each, or four v channels.
        const uint64_t quads = static_cast<uint64_t>(rows) * ((heads + kvHeads) * (headDim / 8) + kvHeads * headDim / 4);
        const auto kernel = splits == 1   ? RopeSplitAppendQuadKernel<1>
                            : splits <= 4 ? RopeSplitAppendQuadKernel<4>
                                          : RopeSplitAppendQuadKernel<kMaxGemmSplits>;
        hipLaunchKernelGGL(kernel, dim3(CeilDiv(quads, 256)), dim3(256), 0, s, qkv, rows, pos0, heads, kvHeads,
                           headDim, maxSeq, ropePow, qhi, qlo, kcache, vcache, splits, bias);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(RopeSplitAppendKernel, dim3(CeilDiv(total, 256)), dim3(256), 0, s, qkv, rows, pos0, heads,
                       kvHeads, headDim, maxSeq, ropePow, qhi, qlo, kcache, vcache, splits, bias);
    return hipGetLastError();
}
}  // namespace muyo

// ------------------------------------------------------------------------------------------------
// C ABI (include/muyo_hip.h).

using namespace muyo;

namespace
{
bool AllAligned16(std::initializer_list<const void*> pointers)
{
    for (const void* p : pointers)
    {
        if (p != nullptr && !Aligned16(p))
        {
            return false;
        }
    }
    return true;
}

int Launched(hipError_t status, const char* name)
{
    return status == hipSuccess ? MUYO_OK : HipStatus(status, name);
}
}  // namespace

extern "C" int muyo_split_f32_f16x2(const float* x, uint64_t count, void* hi, void* lo, void* stream)
{
    const char* name = "split_f32_f16x2";
    if (x == nullptr || hi == nullptr || lo == nullptr)
    {
        return Fail(MUYO_E_NULL, "%s: x, hi and lo are required", name);
    }
    if (count == 0 || count % 4 != 0 || !AllAligned16({x, hi, lo}))
    {
        return Fail(MUYO_E_CONTRACT, "%s: count must be a positive multiple of 4 and the buffers 16-byte aligned",
                    name);
    }
    return Launched(LaunchSplitF32(AsStream(stream), x, count, static_cast<uint16_t*>(hi), static_cast<uint16_t*>(lo)),
                    name);
}

extern "C" int muyo_rms_norm_split_f16x2(const float* x, const float* w, uint32_t rows, uint32_t cols, float eps,
                                         void* hi, void* lo, void* stream)
{
    const char* name = "rms_norm_split_f16x2";
    if (x == nullptr || w == nullptr || hi == nullptr || lo == nullptr)
    {
        return Fail(MUYO_E_NULL, "%s: x, w, hi and lo are required", name);
    }
    if (rows == 0 || cols == 0 || cols % 4 != 0 || !AllAligned16({x, w, hi, lo}))
    {
        return Fail(MUYO_E_CONTRACT, "%s: rows >= 1, cols a positive multiple of 4, buffers 16-byte aligned", name);
    }
    return Launched(LaunchRmsNormSplit(AsStream(stream), x, w, rows, cols, eps, static_cast<uint16_t*>(hi),
                                       static_cast<uint16_t*>(lo)),
                    name);
}

extern "C" int muyo_gemm_split_f16(const void* a_hi, const void* a_lo, const void* w, const float* bias,
                                   const float* residual, float* out, uint32_t rows, uint32_t n, uint32_t k,
                                   void* stream)
{
    const char* name = "gemm_split_f16";
    if (a_hi == nullptr || a_lo == nullptr || w == nullptr || out == nullptr)
    {
        return Fail(MUYO_E_NULL, "%s: a_hi, a_lo, w and out are required", name);
    }
    if (rows == 0 || n == 0 || k == 0 || n % 4 != 0 || k % 8 != 0)
    {
        return Fail(MUYO_E_CONTRACT, "%s: rows >= 1, n a positive multiple of 4, k of 8 (got %u x %u x %u)", name,
                    rows, n, k);
    }
    if (!AllAligned16({a_hi, a_lo, w, bias, residual, out}))
    {
        return Fail(MUYO_E_CONTRACT, "%s: every buffer must be 16-byte aligned", name);
    }
    return Launched(LaunchGemmSplit(AsStream(stream), static_cast<const uint16_t*>(a_hi),
                                    static_cast<const uint16_t*>(a_lo), static_cast<const uint16_t*>(w), bias,
                                    residual, out, rows, n, k),
                    name);
}

extern "C" int muyo_gemm_swiglu_split_f16(const void* a_hi, const void* a_lo, const void* w_gate, const void* w_up,
                                          void* h_hi, void* h_lo, uint32_t rows, uint32_t ffn, uint32_t k,
                                          void* stream)
{
    const char* name = "gemm_swiglu_split_f16";
    if (a_hi == nullptr || a_lo == nullptr || w_gate == nullptr || w_up == nullptr || h_hi == nullptr ||
        h_lo == nullptr)
    {
        return Fail(MUYO_E_NULL, "%s: every buffer is required", name);
    }
    if (rows == 0 || ffn == 0 || k == 0 || ffn % 4 != 0 || k % 8 != 0)
    {
        return Fail(MUYO_E_CONTRACT, "%s: rows >= 1, ffn a positive multiple of 4, k of 8 (got %u x %u x %u)", name,
                    rows, ffn, k);
    }
    if (!AllAligned16({a_hi, a_lo, w_gate, w_up, h_hi, h_lo}))
    {
        return Fail(MUYO_E_CONTRACT, "%s: every buffer must be 16-byte aligned", name);
    }
    return Launched(LaunchGemmSwiGlu(AsStream(stream), static_cast<const uint16_t*>(a_hi),
                                     static_cast<const uint16_t*>(a_lo), static_cast<const uint16_t*>(w_gate),
                                     static_cast<const uint16_t*>(w_up), static_cast<uint16_t*>(h_hi),
                                     static_cast<uint16_t*>(h_lo), rows, ffn, k),
                    name);
}

extern "C" int muyo_rope_split_append_f16kv(const float* qkv, uint32_t rows, int32_t pos0, uint32_t heads,
                                            uint32_t kv_heads, uint32_t head_dim, uint32_t max_seq,
                                            const float* rope_pow, void* q_hi, void* q_lo, void* kcache,
                                            void* vcache, void* stream)
{
    const char* name = "rope_split_append_f16kv";
    if (qkv == nullptr || rope_pow == nullptr || q_hi == nullptr || q_lo == nullptr || kcache == nullptr ||
        vcache == nullptr)
    {
        return Fail(MUYO_E_NULL, "%s: every buffer is required", name);
    }
    if (rows == 0 || heads == 0 || kv_heads == 0 || head_dim == 0 || head_dim % 2 != 0)
    {
        return Fail(MUYO_E_CONTRACT, "%s: rows, heads, kv_heads >= 1 and an even head_dim are required", name);
    }
    if (pos0 < 0 || static_cast<uint64_t>(pos0) + rows > max_seq)
    {
        return Fail(MUYO_E_RANGE, "%s: positions %d..%lld exceed the cache (%u rows)", name, pos0,
                    static_cast<long long>(pos0) + rows - 1, max_seq);
    }
    return Launched(LaunchRopeSplitAppend(AsStream(stream), qkv, rows, pos0, heads, kv_heads, head_dim, max_seq,
                                          rope_pow, static_cast<uint16_t*>(q_hi), static_cast<uint16_t*>(q_lo),
                                          static_cast<uint16_t*>(kcache), static_cast<uint16_t*>(vcache)),
                    name);
}

namespace
{
int CheckPrefillAttentionArgs(const char* name, const void* q_hi, const void* q_lo, const void* kcache,
                              const void* vcache, const void* out_hi, const void* out_lo, uint32_t rows, int32_t pos0,
                              uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t max_seq)
{
    if (q_hi == nullptr || q_lo == nullptr || kcache == nullptr || vcache == nullptr || out_hi == nullptr ||
        out_lo == nullptr)
    {
        return Fail(MUYO_E_NULL, "%s: every buffer is required", name);
    }
    if (rows == 0 || kv_heads == 0 || heads % kv_heads != 0 || heads / kv_heads > 8 ||
        (head_dim != 64 && head_dim != 128))
    {
        return Fail(MUYO_E_UNSUPPORTED, "%s: needs rows >= 1, heads %% kv_heads == 0, group <= 8, head_dim 64 or 128",
                    name);
    }
    if (pos0 < 0 || static_cast<uint64_t>(pos0) + rows > max_seq)
    {
        return Fail(MUYO_E_RANGE, "%s: positions %d..%lld exceed the cache (%u rows)", name, pos0,
                    static_cast<long long>(pos0) + rows - 1, max_seq);
    }
    if (!AllAligned16({q_hi, q_lo, kcache, vcache, out_hi, out_lo}))
    {
        return Fail(MUYO_E_CONTRACT, "%s: every buffer must be 16-byte aligned", name);
    }
    return MUYO_OK;
}
}  // namespace

extern "C" int muyo_prefill_attention_f16kv(const void* q_hi, const void* q_lo, const void* kcache,
                                            const void* vcache, void* out_hi, void* out_lo, uint32_t rows,
                                            int32_t pos0, uint32_t heads, uint32_t kv_heads, uint32_t head_dim,
                                            uint32_t max_seq, float scale, void* stream)
{
    const char* name = "prefill_attention_f16kv";
    const int args = CheckPrefillAttentionArgs(name, q_hi, q_lo, kcache, vcache, out_hi, out_lo, rows, pos0, heads,
                                               kv_heads, head_dim, max_seq);
    if (args != MUYO_OK)
    {
        return args;
    }
    return Launched(LaunchPrefillAttention(AsStream(stream), static_cast<const uint16_t*>(q_hi),
                                           static_cast<const uint16_t*>(q_lo), static_cast<const uint16_t*>(kcache),
                                           static_cast<const uint16_t*>(vcache), static_cast<uint16_t*>(out_hi),
                                           static_cast<uint16_t*>(out_lo), rows, pos0, heads, kv_heads, head_dim,
                                           max_seq, scale),
                    name);
}

extern "C" size_t muyo_prefill_attention_workspace_bytes(uint32_t rows, uint32_t heads, uint32_t head_dim)
{
    if (rows == 0 || heads == 0 || (head_dim != 64 && head_dim != 128))
    {
        return 0;
    }
    return PrefillAttentionWorkspaceFloats(rows, heads, head_dim) * sizeof(float);
}

extern "C" int muyo_prefill_attention_f16kv_ws(const void* q_hi, const void* q_lo, const void* kcache,
                                               const void* vcache, void* out_hi, void* out_lo, uint32_t rows,
                                               int32_t pos0, uint32_t heads, uint32_t kv_heads, uint32_t head_dim,
                                               uint32_t max_seq, float scale, void* workspace,
                                               uint64_t workspace_bytes, void* stream)
{
    const char* name = "prefill_attention_f16kv_ws";
    const int args = CheckPrefillAttentionArgs(name, q_hi, q_lo, kcache, vcache, out_hi, out_lo, rows, pos0, heads,
                                               kv_heads, head_dim, max_seq);
    if (args != MUYO_OK)
    {
        return args;
    }
    const size_t floats = PrefillAttentionWorkspaceFloats(rows, heads, head_dim);
    if (workspace == nullptr || !Aligned16(workspace) || workspace_bytes < floats * sizeof(float))
    {
        return Fail(MUYO_E_CONTRACT, "%s: needs a 16-byte aligned workspace of %zu bytes (got %llu)", name,
                    floats * sizeof(float), static_cast<unsigned long long>(workspace_bytes));
    }
    return Launched(LaunchPrefillAttention(AsStream(stream), static_cast<const uint16_t*>(q_hi),
                                           static_cast<const uint16_t*>(q_lo), static_cast<const uint16_t*>(kcache),
                                           static_cast<const uint16_t*>(vcache), static_cast<uint16_t*>(out_hi),
                                           static_cast<uint16_t*>(out_lo), rows, pos0, heads, kv_heads, head_dim,
                                           max_seq, scale, static_cast<float*>(workspace), floats),
                    name);
}
