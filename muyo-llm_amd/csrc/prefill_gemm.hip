// Split-f16 GEMMs of the batched prefill: out[m][n] = sum_k (ahi + alo)[m][k] * W[n][k] on
// v_mfma_f32_32x32x16_f16, with fused epilogues.
//
// The weights are the matrix core's A operand (rows n), the activation planes its B operand
// (columns m), so a lane ends with four consecutive n of one m per accumulator group: 16-byte
// stores into row-major [m][n]. Each weight fragment meets the hi and the lo plane.
#include <algorithm>
#include <cmath>
#include <limits>

#include "prefill.hpp"
#include "prefill_core.hpp"

namespace muyo
{
namespace
{
/// K is split on multiples of this many columns (the widest K slab of a tile shape).
constexpr uint32_t kGemmSplitUnit = 128;

/// out = acc + bias[n] + residual[m][n] (either may be null); virtual rows are the weight rows.
/// With `partial` each K split z stores its raw sums to plane z of `partial` ([splits][rows][n]);
/// bias and residual are then the consumer's to add.
struct PlainEpi
{
    const uint16_t* w;
    const float* bias;
    const float* residual;
    float* out;
    uint32_t n, k;
    float* partial = nullptr;

    /// LDS row that holds virtual row v of a 32-row block.
    __device__ static uint32_t LdsRow(uint32_t v) { return v; }
    /// The matrix row in LDS row u (uniform; clamped to the last row), and whether u + r exists.
    __device__ const uint16_t* Row(uint32_t u) const { return w + static_cast<uint64_t>(min(u, n - 1)) * k; }
    __device__ bool Live(uint32_t u, uint32_t r) const { return u + r < n; }

    template <int kNb, int kMb>
    __device__ void Finish(const floatx16 (&acc)[kNb][kMb], uint32_t n0, uint32_t m0, uint32_t rows, uint32_t z) const
    {
        const uint32_t lane = threadIdx.x % kWave;
        const uint32_t h = lane / 32;
#pragma unroll
        for (int mb = 0; mb < kMb; ++mb)
        {
            const uint32_t m = m0 + mb * 32 + lane % 32;
            if (m >= rows)
            {
                continue;
            }
#pragma unroll
            for (int nb = 0; nb < kNb; ++nb)
            {
#pragma unroll
                for (int g = 0; g < 4; ++g)
                {
                    const uint32_t nn = n0 + nb * 32 + 8 * g + 4 * h;
                    if (nn >= n)
                    {
                        continue;
                    }
                    float4 v = make_float4(acc[nb][mb][4 * g], acc[nb][mb][4 * g + 1], acc[nb][mb][4 * g + 2],
                                           acc[nb][mb][4 * g + 3]);
                    const uint64_t at = static_cast<uint64_t>(m) * n + nn;
                    if (partial != nullptr)
                    {
                        *reinterpret_cast<float4*>(partial + static_cast<uint64_t>(z) * rows * n + at) = v;
                        continue;
                    }
                    if (bias != nullptr)
                    {
                        const float4 b = *reinterpret_cast<const float4*>(bias + nn);
                        v.x += b.x;
                        v.y += b.y;
                        v.z += b.z;
                        v.w += b.w;
                    }
                    if (residual != nullptr)
                    {
                        const float4 r = *reinterpret_cast<const float4*>(residual + at);
                        v.x = r.x + v.x;
                        v.y = r.y + v.y;
                        v.z = r.z + v.z;
                        v.w = r.w + v.w;
                    }
                    *reinterpret_cast<float4*>(out + at) = v;
                }
            }
        }
    }
};

/// Gate and up interleaved eight rows at a time, so that any 32-row block is complete: virtual
/// rows 16 t + j are gate row 8 t + j for j < 8 and up row 8 t + j - 8 for the other eight. A lane
/// then holds g (accumulator groups 0 and 2) and u (1 and 3) of the same (m, f) and writes
/// silu(g) * u (swiglu.comp's op) as split planes. In LDS a block's 16 gate rows come first, so
/// that the rows one load instruction brings are neighbours in one matrix.
struct SwiGluEpi
{
    const uint16_t* gate;
    const uint16_t* up;
    uint16_t* hhi;
    uint16_t* hlo;
    uint32_t ffn, k;

    __device__ static uint32_t LdsRow(uint32_t v) { return (v & 8u) * 2 + (v >> 4) * 8 + (v & 7u); }
    __device__ static uint32_t First(uint32_t u) { return u / 32 * 16 + u % 16; }
    __device__ const uint16_t* Row(uint32_t u) const
    {
        return (u % 32 < 16 ? gate : up) + static_cast<uint64_t>(min(First(u), ffn - 1)) * k;
    }
    __device__ bool Live(uint32_t u, uint32_t r) const { return First(u) + r < ffn; }

    template <int kNb, int kMb>
    __device__ void Finish(const floatx16 (&acc)[kNb][kMb], uint32_t n0, uint32_t m0, uint32_t rows, uint32_t) const
    {
        const uint32_t lane = threadIdx.x % kWave;
        const uint32_t h = lane / 32;
#pragma unroll
        for (int mb = 0; mb < kMb; ++mb)
        {
            const uint32_t m = m0 + mb * 32 + lane % 32;
            if (m >= rows)
            {
                continue;
            }
#pragma unroll
            for (int nb = 0; nb < kNb; ++nb)
            {
#pragma unroll
                for (int g = 0; g < 4; g += 2)
                {
                    const uint32_t f = (n0 + nb * 32) / 2 + 4 * g + 4 * h;
                    if (f >= ffn)
                    {
                        continue;
                    }
                    float a[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                    {
                        const float gv = acc[nb][mb][4 * g + t];
                        a[t] = gv / (1.0f + expf(-gv)) * acc[nb][mb][4 * g + 4 + t];
                    }
                    StoreSplit4(hhi, hlo, static_cast<uint64_t>(m) * ffn + f, a[0], a[1], a[2], a[3]);
                }
            }
        }
    }
};

/// A tile of kBm tokens x kBn weight rows by kWm x kWn x kWk waves: a wave owns kMb x kNb blocks
/// of 32 x 32 outputs, and with kWk > 1 that many waves own the same blocks and every kWk-th step
/// of 16 columns, their sums meeting in LDS at the end.
///
/// K advances kBk columns at a time through kStages LDS buffers. The loads go from memory to LDS
/// without passing through registers (LoadToLds), up to kStages - 1 slabs ahead, and a slab costs
/// one barrier: past it, every wave's part of the slab has arrived and every wave is done with the
/// buffer that the next loads overwrite. WaitAndMeet counts the loads (a wave's complete in order,
/// kLoads a slab). Rows are not padded (the load writes 1 KB at a stretch), so each row's 16-byte
/// chunks are permuted by the row number instead, on the global side of the load; the fragment
/// reads of eight consecutive rows then touch no bank twice. (The 16 that share the 64 banks still
/// meet in pairs. A permutation without that, 4.0 conflict cycles per LDS instruction cycle less,
/// left the GEMMs within 0.4 % and whole prompts of 613 rows 2 % slower by its address
/// instructions: waves wait on LDS 2 to 6 % of their cycles.)
///
/// What bounds it. With random data the matrix cores alone sustain 1.67 PFLOP/s on this part (its
/// power limit; 2.3 with zeros), and 1.5 with an LDS fragment read for every two operations. Loads
/// from L2 run at 34 TB/s but anything past it at 7, so what every XCD has to fetch counts
/// (GemmOrder). A single wave per SIMD leaves the matrix cores idle between a barrier and its first
/// fragments: the shapes have two (or two workgroups per CU) where LDS allows.
/// Measured at the unsplit entry points, before (a register-staged kernel, one LDS buffer) and now,
/// us: 0.5B gate+up 301 rows 29 / 18.0, 613 rows 41 / 30.4, 2048 rows 94 / 94; down 301 rows
/// 82 / 22.4, 2048 rows 85 / 51; q|k|v 613 rows 21 / 10.0; 7B gate+up 45 rows 99 / 65, 2048 rows
/// 1054 / 990; down 45 rows 308 / 84, 2048 rows 621 / 549; o_proj 2048 rows 123 / 111; q|k|v
/// 2048 rows 194 / 156.
template <int kWm, int kWn, int kWk, int kMb, int kNb, int kStages, int kBk, int kPerCu>
struct GemmTile
{
    static constexpr int kWaves = kWm * kWn * kWk;
    static constexpr int kThreads = kWave * kWaves;
    static constexpr int kBm = 32 * kMb * kWm;
    static constexpr int kBn = 32 * kNb * kWn;
    static constexpr int kRows = 2 * kBm + kBn;           // LDS rows of a slab: hi, lo, weights
    static constexpr int kRowBytes = 2 * kBk;
    static constexpr int kChunks = kBk / 8;               // 16-byte chunks per row
    static constexpr int kRowsPerLoad = kWave / kChunks;  // rows one load instruction brings
    static constexpr int kGroups = kRows / kRowsPerLoad;
    static constexpr int kLoads = kGroups / kWaves;       // per wave and slab
    static constexpr int kStageBytes = kRows * kRowBytes;
    static constexpr int kSteps = kBk / 16 / kWk;         // per wave and slab
    static constexpr int kMinWaves = (kWaves * kPerCu + 3) / 4;  // per SIMD
    static constexpr int kMaxBlocks = kPerCu;             // workgroups a CU holds (by LDS)
    static constexpr bool kLowSums = kMb * kNb <= 4;      // two sums per block
    static constexpr int kSumFloats = 1024 * kNb * kMb;   // a wave's tile
    static_assert(kRows % kRowsPerLoad == 0 && kBm % kRowsPerLoad == 0 && 16 % kRowsPerLoad == 0, "row groups");
    static_assert(kGroups % kWaves == 0, "every wave has as many loads in flight as WaitAndMeet counts");
    static_assert(kBk % (16 * kWk) == 0 && kGemmSplitUnit % kBk == 0, "steps");
    static_assert(kStages >= 2 && kStages <= 5 && kStages * kStageBytes * kPerCu <= 160 * 1024, "LDS");
    static_assert((kWk - 1) * kWm * kWn * kSumFloats * 4 <= kStages * kStageBytes, "LDS of the K sums");
};

/// This workgroup's tile and K split. Workgroups are dealt to the 8 XCDs round-robin by id; with
/// the renumbering XCD x runs the x-th eighth of one sequence: the splits, in each the groups of
/// `group` token tiles, in each the weight tiles, in each the group's token tiles. (The results do
/// not depend on where a workgroup runs.)
///
/// What an XCD's resident workgroups read of a slab comes from past its L2 once: the rows of the
/// group's token tiles and of the weight tiles beside them, the fewest when the two are about as
/// many (GroupTiles has the rule). With all token tiles in a group instead (or all weight tiles, where the
/// activations were the larger operand), 8192 rows of 14336 x 4096 gate+up took 3.92 ms, with groups
/// of four 256-row tiles 3.14; 2048 rows of 4864 x 896 on 128 x 256 tiles 95.4 / 93.1 us, 8192 rows
/// of 3584 x 3584 383 / 350.
struct GemmOrder
{
    uint32_t mTiles, nTiles, group;

    __device__ void Tile(uint32_t& mt, uint32_t& nt, uint32_t& z) const
    {
        const uint32_t xcd = blockIdx.x % 8;
        const uint32_t id = xcd * (gridDim.x / 8) + min(xcd, gridDim.x % 8) + blockIdx.x / 8;
        const uint32_t plane = mTiles * nTiles;
        z = id / plane;
        const uint32_t t = id % plane;
        const uint32_t first = t / (group * nTiles) * group;
        const uint32_t width = min(group, mTiles - first);
        mt = first + t % (group * nTiles) % width;
        nt = t % (group * nTiles) / width;
    }
};

template <typename T, int kWm, int kWn, int kWk, int kMb, int kNb, int kStages, int kBk, typename Epi>
__global__ __launch_bounds__(T::kThreads, T::kMinWaves) void GemmSplitKernel(const uint16_t* __restrict__ ahi,
                                                                             const uint16_t* __restrict__ alo, Epi epi,
                                                                             uint32_t rows, uint32_t k,
                                                                             uint32_t kPerSplit, GemmOrder order)
{
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kStages * T::kStageBytes];
    constexpr uint32_t kAGroups = 2 * T::kBm / T::kRowsPerLoad;

    const uint32_t lane = threadIdx.x % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    uint32_t mt, nt, z;
    order.Tile(mt, nt, z);
    const uint32_t m0 = mt * T::kBm;
    const uint32_t n0 = nt * T::kBn;
    const uint32_t kBegin = z * kPerSplit;
    const uint32_t kEnd = min(k, kBegin + kPerSplit);
    const uint32_t slabs = kBegin < kEnd ? (kEnd - kBegin + kBk - 1) / kBk : 0;

    // Load i of a wave brings LDS rows [g * kRowsPerLoad, ...) of a slab. The address is a row
    // group's, uniform across the wave, plus the lane's offset. A lane whose row lies past the
    // matrix reads the group's first row (clamped to the last) instead, and one whose chunk lies
    // past kEnd the row's first chunk of the slab: in bounds, and either not stored or zeroed
    // below.
    const uint32_t groupRow = lane / T::kChunks;
    const uint32_t ldsBase =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds));
    auto load = [&](uint32_t stage, uint32_t k0, int i)
    {
        const uint32_t g = wave + i * T::kWaves;
        const uint32_t r = g * T::kRowsPerLoad;
        const uint32_t row = r + groupRow;
        const uint32_t chunk = (lane % T::kChunks) ^ (kBk == 32 ? (row >> 1) & 3u : row & 7u);
        const uint32_t first = (k0 + (k0 + chunk * 8 < kEnd ? chunk * 8 : 0u)) * 2;
        const uint16_t* base;
        bool live;
        if (g < kAGroups)
        {
            const bool lo = r >= T::kBm;
            const uint32_t m = m0 + (lo ? r - T::kBm : r);
            base = (lo ? alo : ahi) + static_cast<uint64_t>(min(m, rows - 1)) * k;
            live = m + groupRow < rows;
        }
        else
        {
            const uint32_t u = n0 + r - 2 * T::kBm;
            base = epi.Row(u);
            live = epi.Live(u, groupRow);
        }
        const uint32_t offset = live ? first + groupRow * k * 2 : first;
        LoadToLds(ldsBase + stage * T::kStageBytes + wave * 1024, i * T::kWaves * 1024, offset, base);
    };

    const uint32_t kg = wave / (kWm * kWn);
    const uint32_t wm = wave / kWn % kWm;
    const uint32_t wn = wave % kWn;
    const uint32_t h = lane / 32;
    const uint32_t aRow = lane % 32;
    const uint32_t wRow = Epi::LdsRow(lane % 32);
    const uint32_t aSwizzle = kBk == 32 ? (aRow >> 1) & 3u : aRow & 7u;
    const uint32_t wSwizzle = kBk == 32 ? (wRow >> 1) & 3u : wRow & 7u;

    // The lo products (2^-11 of the hi products) have sums of their own where the registers allow:
    // half as many roundings at the size of the result.
    floatx16 acc[kNb][kMb];
    floatx16 low[T::kLowSums ? kNb : 1][T::kLowSums ? kMb : 1];
#pragma unroll
    for (int a = 0; a < kNb; ++a)
    {
#pragma unroll
        for (int b = 0; b < kMb; ++b)
        {
            acc[a][b] = floatx16{};
            if constexpr (T::kLowSums)
            {
                low[a][b] = floatx16{};
            }
        }
    }
#pragma unroll
    for (uint32_t s = 0; s < kStages - 1; ++s)
    {
        if (s < slabs)
        {
#pragma unroll
            for (int i = 0; i < T::kLoads; ++i)
            {
                load(s, kBegin + s * kBk, i);
            }
        }
    }
    uint32_t stage = 0;
    for (uint32_t s = 0; s < slabs; ++s)
    {
        // The slabs after this one that are already requested stay in flight.
        const uint32_t ahead = min(static_cast<uint32_t>(kStages - 2), slabs - 1 - s);
        if (kStages <= 2 || ahead == 0)
        {
            WaitAndMeet<0>();
        }
        else if (kStages == 3 || ahead == 1)
        {
            WaitAndMeet<T::kLoads>();
        }
        else if (kStages == 4 || ahead == 2)
        {
            WaitAndMeet<2 * T::kLoads>();
        }
        else
        {
            WaitAndMeet<3 * T::kLoads>();
        }
        const bool more = s + kStages - 1 < slabs;
        const uint32_t freed = stage == 0 ? kStages - 1 : stage - 1;
        const uint8_t* tile = lds + stage * T::kStageBytes;
#pragma unroll
        for (int q = 0; q < T::kSteps; ++q)
        {
            const uint32_t step = q * kWk + kg;
            const uint32_t aAt = ((step * 2 + h) ^ aSwizzle) * 16 + aRow * T::kRowBytes;
            const uint32_t wAt = ((step * 2 + h) ^ wSwizzle) * 16 + wRow * T::kRowBytes;
            half8 wf[kNb], xh[kMb], xl[kMb];
#pragma unroll
            for (int b = 0; b < kNb; ++b)
            {
                wf[b] = *reinterpret_cast<const half8*>(tile + (2 * T::kBm + (wn * kNb + b) * 32) * T::kRowBytes + wAt);
            }
#pragma unroll
            for (int b = 0; b < kMb; ++b)
            {
                const uint8_t* x = tile + (wm * kMb + b) * 32 * T::kRowBytes + aAt;
                xh[b] = *reinterpret_cast<const half8*>(x);
                xl[b] = *reinterpret_cast<const half8*>(x + T::kBm * T::kRowBytes);
            }
            if (s + 1 == slabs && kBegin + s * kBk + step * 16 + 8 * h >= kEnd)
            {
#pragma unroll
                for (int b = 0; b < kNb; ++b)
                {
                    wf[b] = half8{};
                }
#pragma unroll
                for (int b = 0; b < kMb; ++b)
                {
                    xh[b] = half8{};
                    xl[b] = half8{};
                }
            }
            // The hi products of every block, then the lo products, so that independent
            // matrix-core operations separate two that accumulate into the same block.
#pragma unroll
            for (int a = 0; a < kNb; ++a)
            {
#pragma unroll
                for (int b = 0; b < kMb; ++b)
                {
                    acc[a][b] = Mfma(wf[a], xh[b], acc[a][b]);
                }
            }
            // A step's share of the loads, spread over the slab: issued at once, they would hold
            // the wave at the address unit before its first product.
            if (more)
            {
#pragma unroll
                for (int i = q * T::kLoads / T::kSteps; i < (q + 1) * T::kLoads / T::kSteps; ++i)
                {
                    load(freed, kBegin + (s + kStages - 1) * kBk, i);
                }
            }
#pragma unroll
            for (int a = 0; a < kNb; ++a)
            {
#pragma unroll
                for (int b = 0; b < kMb; ++b)
                {
                    if constexpr (T::kLowSums)
                    {
                        low[a][b] = Mfma(wf[a], xl[b], low[a][b]);
                    }
                    else
                    {
                        acc[a][b] = Mfma(wf[a], xl[b], acc[a][b]);
                    }
                }
            }
        }
        stage = stage + 1 == kStages ? 0 : stage + 1;
    }
    if constexpr (T::kLowSums)
    {
#pragma unroll
        for (int a = 0; a < kNb; ++a)
        {
#pragma unroll
            for (int b = 0; b < kMb; ++b)
            {
                acc[a][b] += low[a][b];
            }
        }
    }
    if constexpr (kWk > 1)
    {
        // K groups 1.. leave their tiles in LDS (done with as slabs), group 0 adds them in order.
        __syncthreads();
        float* sums = reinterpret_cast<float*>(lds);
        if (kg > 0)
        {
            float* to = sums + (wave - kWm * kWn) * T::kSumFloats + lane * 4;
#pragma unroll
            for (int a = 0; a < kNb; ++a)
            {
#pragma unroll
                for (int b = 0; b < kMb; ++b)
                {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                    {
                        *reinterpret_cast<float4*>(to + ((a * kMb + b) * 4 + q) * 256) =
                            make_float4(acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2],
                                        acc[a][b][4 * q + 3]);
                    }
                }
            }
        }
        __syncthreads();
        if (kg > 0)
        {
            return;
        }
#pragma unroll 1
        for (int other = 0; other < kWk - 1; ++other)
        {
            const float* from = sums + (other * kWm * kWn + wave) * T::kSumFloats + lane * 4;
#pragma unroll
            for (int a = 0; a < kNb; ++a)
            {
#pragma unroll
                for (int b = 0; b < kMb; ++b)
                {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                    {
                        const float4 v = *reinterpret_cast<const float4*>(from + ((a * kMb + b) * 4 + q) * 256);
                        acc[a][b][4 * q] += v.x;
                        acc[a][b][4 * q + 1] += v.y;
                        acc[a][b][4 * q + 2] += v.z;
                        acc[a][b][4 * q + 3] += v.w;
                    }
                }
            }
        }
    }
    epi.Finish(acc, n0 + wn * 32 * kNb, m0 + wm * 32 * kMb, rows, z);
}

/// The tile shapes, X(index, waves m, n, k, blocks m, n, LDS stages, K slab, workgroups per CU).
/// Eight of 25 that were measured over the prefill's GEMMs (both models' four matrices and 14 more,
/// 1 to 8192 rows, every K split): with these eight the best choice per GEMM is within 0.5 % of the
/// best of the 14 shapes measured last on average.
#define MUYO_GEMM_TILES(X)         \
    X(0, 4, 2, 1, 2, 4, 3, 32, 1)  \
    X(1, 2, 2, 2, 2, 3, 2, 64, 1)  \
    X(2, 2, 4, 1, 2, 2, 3, 32, 1)  \
    X(3, 2, 4, 1, 1, 2, 3, 64, 1)  \
    X(4, 2, 2, 2, 1, 3, 4, 64, 1)  \
    X(5, 1, 2, 2, 1, 2, 3, 64, 2)  \
    X(6, 1, 2, 4, 1, 2, 3, 128, 1) \
    X(7, 1, 1, 4, 1, 2, 3, 128, 1)

/// What the choice of a shape needs to know. slabUs is the time of 64 columns of K with the CUs
/// busy, tileUs what a round of tiles costs besides (first loads, epilogue), both fitted to those
/// measurements. `margin` is above 1 for the shapes without sums for the lo products, which round
/// twice as often: they are taken where they gain more than that.
struct GemmTileCost
{
    uint32_t bm, bn, bk, stages, perCu;
    double slabUs, tileUs, margin;
};

constexpr GemmTileCost kGemmTiles[] = {
    {256, 256, 32, 3, 1, 2.547, 0.01, 1.12}, {128, 192, 64, 2, 1, 1.495, 0.17, 1.03},
    {128, 256, 32, 3, 1, 1.753, 0.01, 1.0},  {64, 256, 64, 3, 1, 0.941, 0.02, 1.0},
    {64, 192, 64, 4, 1, 0.744, 0.72, 1.0},   {32, 128, 64, 3, 2, 0.756, 0.08, 1.0},
    {32, 128, 128, 3, 1, 0.380, 2.05, 1.0},  {32, 64, 128, 3, 1, 0.292, 2.03, 1.0},
};
constexpr int kGemmTileCount = sizeof(kGemmTiles) / sizeof(kGemmTiles[0]);
constexpr uint32_t kCus = 256;

/// Columns of K per split.
uint32_t ColumnsPerSplit(uint32_t k, uint32_t splits)
{
    return CeilDiv(CeilDiv(k, kGemmSplitUnit), splits) * kGemmSplitUnit;
}

/// Token tiles of a group of GemmOrder. Over several rounds an XCD's 32 CUs hold about as many rows of
/// both planes as of weights, in groups of about the same size. In a single round all tiles are
/// resident, and an XCD's eighth of them is left in whole columns or rows of tiles: every token tile
/// in one group, or one to a group where the activations are the larger operand (32 x 128 tiles, us,
/// groups by the rule above / so: 513 rows of gate+up 2000 x 1784 26.8 / 21.9, 1500 rows of
/// 896 x 4864 46.5 / 44.7, 1300 rows of 1000 x 1784 27.8 / 25.1).
uint32_t GroupTiles(const GemmTileCost& tile, uint32_t rows, uint32_t n, uint32_t splits)
{
    const uint32_t mTiles = CeilDiv(rows, tile.bm);
    if (static_cast<uint64_t>(mTiles) * CeilDiv(n, tile.bn) * splits <= kCus * tile.perCu)
    {
        return static_cast<uint64_t>(rows) * 2 <= n ? mTiles : 1;
    }
    const double most = std::round(std::sqrt(kCus / 8.0 * tile.perCu * tile.bn / (2.0 * tile.bm)));
    return CeilDiv(mTiles, CeilDiv(mTiles, static_cast<uint32_t>(most)));
}

/// Estimated us of a launch of `tile` over `splits` K splits: the rounds of resident workgroups
/// times their slabs, or the time the weights take to arrive with the bytes each round keeps in
/// flight (1.52 us each, at most 9 TB/s), whichever is longer; the result's way to memory; and with
/// splits the partial planes' and their consumer's. It ranks the shapes: over the measured GEMMs
/// (unsplit with weights in cache and from memory, split with weights from memory, as a prompt's
/// layers find them) the chosen one was 0.7 % slower than the fastest of the eight on average, 15 %
/// at most. (Fitted with weights in cache alone, it left long K unsplit at 800 rows: 896 x 4864
/// 24.4 us there, 33.9 in a prompt, where three splits take 25.4.)
double GemmCost(const GemmTileCost& tile, uint32_t rows, uint32_t n, uint32_t k, uint32_t splits)
{
    const double tiles = static_cast<double>(CeilDiv(rows, tile.bm)) * CeilDiv(n, tile.bn) * splits;
    const double slots = static_cast<double>(kCus) * tile.perCu;
    const double fullRounds = std::floor(tiles / slots);
    const double last = tiles - fullRounds * slots;
    const double rounds = fullRounds + (last > 0.0 ? 1.0 : 0.0);
    const double slabs = std::min(CeilDiv(k, 64), ColumnsPerSplit(k, splits) / 64);
    // A CU's workgroups slow one another: in one round, as many as meet another.
    const double shared = fullRounds > 0.0 ? 1.0 : std::max(tiles - kCus, 0.0) / kCus;
    const double slow = tile.perCu > 1 ? 0.98 + 0.02 * shared : 1.0;
    const double tileBytes = 2.0 * n * k / tiles;
    const double inFlight = static_cast<double>(tile.stages - 1) * tile.bn * tile.bk * 2;
    auto arrive = [&](double count) { return count * tileBytes / std::min(9.09e6, count * inFlight / 1.52); };
    const double weights = fullRounds * arrive(slots) + (last > 0.0 ? arrive(last) : 0.0);
    const double us = std::max(rounds * (slabs * tile.slabUs * slow + tile.tileUs), weights + tile.tileUs);
    const double values = static_cast<double>(rows) * n / 1.0e6;
    return tile.margin * (2.0 + us + 1.70 * values) + (splits > 1 ? 14.57 / 4.0 * splits * values : 0.0);
}

/// The fastest shape by that estimate.
int BestTile(uint32_t rows, uint32_t n, uint32_t k, uint32_t splits)
{
    int best = 0;
    for (int i = 1; i < kGemmTileCount; ++i)
    {
        if (GemmCost(kGemmTiles[i], rows, n, k, splits) < GemmCost(kGemmTiles[best], rows, n, k, splits))
        {
            best = i;
        }
    }
    return best;
}

template <typename Epi>
hipError_t LaunchGemm(hipStream_t s, const uint16_t* ahi, const uint16_t* alo, const Epi& epi, uint32_t rows,
                      uint32_t virtualRows, uint32_t k, uint32_t splits = 1)
{
    if (rows == 0 || virtualRows == 0 || k == 0 || splits == 0)
    {
        return hipErrorInvalidValue;
    }
    const int best = BestTile(rows, virtualRows, k, splits);
    const GemmOrder order{CeilDiv(rows, kGemmTiles[best].bm), CeilDiv(virtualRows, kGemmTiles[best].bn),
                          GroupTiles(kGemmTiles[best], rows, virtualRows, splits)};
    const uint64_t blocks = static_cast<uint64_t>(order.mTiles) * order.nTiles * splits;
    if (blocks > std::numeric_limits<int32_t>::max())
    {
        return hipErrorInvalidValue;
    }
    const uint32_t kPerSplit = ColumnsPerSplit(k, splits);
    switch (best)
    {
#define MUYO_GEMM_LAUNCH(I, WM, WN, WK, MB, NB, ST, BK, PER)                                                           \
    case I:                                                                                                            \
    {                                                                                                                  \
        using T = GemmTile<WM, WN, WK, MB, NB, ST, BK, PER>;                                                           \
        static_assert(T::kBm == kGemmTiles[I].bm && T::kBn == kGemmTiles[I].bn && BK == kGemmTiles[I].bk &&            \
                          ST == kGemmTiles[I].stages && PER == kGemmTiles[I].perCu &&                                  \
                          T::kLowSums == (kGemmTiles[I].margin == 1.0),                                                \
                      "kGemmTiles");                                                                                   \
        hipLaunchKernelGGL((GemmSplitKernel<T, WM, WN, WK, MB, NB, ST, BK, Epi>), dim3(static_cast<uint32_t>(blocks)), \
                           dim3(T::kThreads), 0, s, ahi, alo, epi, rows, k, kPerSplit, order);                         \
        break;                                                                                                         \
    }
        MUYO_GEMM_TILES(MUYO_GEMM_LAUNCH)
#undef MUYO_GEMM_LAUNCH
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
}  // namespace

uint32_t GemmSplits(uint32_t rows, uint32_t n, uint32_t k)
{
    uint32_t best = 1;
    double bestCost = std::numeric_limits<double>::infinity();
    for (uint32_t splits = 1; splits <= MaxGemmSplits(rows) && rows > 0 && n > 0 && k > 0; ++splits)
    {
        // Splits of whole kGemmSplitUnits, none of them empty.
        if (CeilDiv(k, ColumnsPerSplit(k, splits)) != splits)
        {
            continue;
        }
        const double cost = GemmCost(kGemmTiles[BestTile(rows, n, k, splits)], rows, n, k, splits);
        if (cost < bestCost)
        {
            bestCost = cost;
            best = splits;
        }
    }
    return best;
}

hipError_t LaunchGemmSplit(hipStream_t s, const uint16_t* ahi, const uint16_t* alo, const uint16_t* w,
                           const float* bias, const float* residual, float* out, uint32_t rows, uint32_t n,
                           uint32_t k, float* partial, uint32_t splits)
{
    if (n % 4 != 0 || k % 8 != 0 || splits == 0 || splits > kMaxGemmSplits || (splits > 1 && partial == nullptr))
    {
        return hipErrorInvalidValue;
    }
    PlainEpi epi{w, bias, residual, out, n, k};
    epi.partial = splits > 1 ? partial : nullptr;
    return LaunchGemm(s, ahi, alo, epi, rows, n, k, splits);
}

hipError_t LaunchGemmSwiGlu(hipStream_t s, const uint16_t* ahi, const uint16_t* alo, const uint16_t* wgate,
                            const uint16_t* wup, uint16_t* hhi, uint16_t* hlo, uint32_t rows, uint32_t ffn,
                            uint32_t k)
{
    if (ffn % 4 != 0 || k % 8 != 0)
    {
        return hipErrorInvalidValue;
    }
    // Two virtual rows (gate, up) per output, in whole 32-row blocks.
    const uint32_t virtualRows = 2 * CeilDiv(ffn, 16) * 16;
    return LaunchGemm(s, ahi, alo, SwiGluEpi{wgate, wup, hhi, hlo, ffn, k}, rows, virtualRows, k);
}
}  // namespace muyo

// For the tests (no device needed): the tile (tokens, weight rows, columns of a slab), token tiles
// per group, and K splits of a launch; splits 0 for the decoder's choice of them. For the swiglu
// GEMM n is twice the outputs, in whole 32s.
extern "C" void muyo_prefill_gemm_plan(uint32_t rows, uint32_t n, uint32_t k, uint32_t splits, uint32_t plan[5])
{
    const uint32_t z = splits > 0 ? splits : muyo::GemmSplits(rows, n, k);
    const muyo::GemmTileCost& tile = muyo::kGemmTiles[muyo::BestTile(rows, n, k, z)];
    plan[0] = tile.bm;
    plan[1] = tile.bn;
    plan[2] = tile.bk;
    plan[3] = muyo::GroupTiles(tile, rows, n, z);
    plan[4] = z;
}
