// Causal flash attention of the batched prefill over the fp16 cache.
#include <algorithm>
#include <cmath>
#include <limits>
#include <type_traits>

#include "prefill.hpp"
#include "prefill_core.hpp"

namespace muyo
{
namespace
{
typedef short short4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

constexpr int kAttnStep = 64;  // keys of one step: an LDS buffer of K and V rows
constexpr int kAttnWaves = 4;  // a workgroup's; two workgroups fit a CU

/// Key tiles of 32 that a query tile attends to: cache rows 0 .. its last query's position.
__host__ __device__ inline uint32_t AttnKeyTiles(uint32_t qtile, uint32_t rows, int32_t pos0)
{
    const uint32_t last = qtile * 32 + 31 < rows ? qtile * 32 + 31 : rows - 1;
    return (static_cast<uint32_t>(pos0) + last) / 32 + 1;
}

/// Softmax partials of the chunks of split tiles: [kAttnMaxChunks][rows][heads] (running max in
/// log2 units, sum) and [kAttnMaxChunks][rows][heads][headDim] (unnormalised P.V).
struct AttnPartials
{
    float* max;
    float* sum;
    float* acc;
};

/// Combines the chunk partials of the split tiles' queries into their output planes: out = sum_c
/// 2^(m_c - M) acc_c / sum_c 2^(m_c - M) l_c, M the largest m_c (a chunk with no key of the query
/// weighs 0). A thread per (query, head, 4 channels); queries of unsplit tiles are left alone.
__global__ __launch_bounds__(256) void PrefillAttnMergeKernel(AttnPartials part, uint16_t* __restrict__ ohi,
                                                              uint16_t* __restrict__ olo, uint32_t rows, int32_t pos0,
                                                              uint32_t heads, uint32_t headDim, uint32_t chunkTiles)
{
    const uint32_t quads = headDim / 4;
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<uint64_t>(rows) * heads * quads)
    {
        return;
    }
    const uint32_t channel = static_cast<uint32_t>(i % quads) * 4;
    const uint32_t head = static_cast<uint32_t>(i / quads % heads);
    const uint32_t m = static_cast<uint32_t>(i / quads / heads);
    const uint32_t keyTiles = AttnKeyTiles(m / 32, rows, pos0);
    if (keyTiles <= chunkTiles)
    {
        return;
    }
    const uint32_t chunks = (keyTiles + chunkTiles - 1) / chunkTiles;
    // Every slot's operands requested at once (slots past `chunks` reread slot 0 and weigh 0).
    float mc[kAttnMaxChunks];
    float lc[kAttnMaxChunks];
    float4 ac[kAttnMaxChunks];
#pragma unroll
    for (uint32_t c = 0; c < kAttnMaxChunks; ++c)
    {
        const uint64_t at = (static_cast<uint64_t>(c < chunks ? c : 0) * rows + m) * heads + head;
        mc[c] = part.max[at];
        lc[c] = part.sum[at];
        ac[c] = *reinterpret_cast<const float4*>(part.acc + at * headDim + channel);
    }
    float top = -INFINITY;
#pragma unroll
    for (uint32_t c = 0; c < kAttnMaxChunks; ++c)
    {
        top = c < chunks ? fmaxf(top, mc[c]) : top;
    }
    float den = 0.0f;
    float4 num = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (uint32_t c = 0; c < kAttnMaxChunks; ++c)
    {
        if (c < chunks)
        {
            const float w = mc[c] == -INFINITY ? 0.0f : exp2f(mc[c] - top);
            den = fmaf(w, lc[c], den);
            num.x = fmaf(w, ac[c].x, num.x);
            num.y = fmaf(w, ac[c].y, num.y);
            num.z = fmaf(w, ac[c].z, num.z);
            num.w = fmaf(w, ac[c].w, num.w);
        }
    }
    const float inv = 1.0f / den;
    StoreSplit4(ohi, olo, static_cast<uint64_t>(m) * heads * headDim + head * headDim + channel, num.x * inv,
                num.y * inv, num.z * inv, num.w * inv);
}

/// hi and lo planes of eight softmax weights, as the matrix core's B operand: hi rounded to f16,
/// lo the rest rounded to f16.
__device__ __forceinline__ void SplitWeights(const float* p, half8& hi, half8& lo)
{
    uint4v h, l;
#pragma unroll
    for (int v = 0; v < 4; ++v)
    {
        const float2v two = {p[2 * v], p[2 * v + 1]};
        const uint32_t bits = __builtin_bit_cast(uint32_t, __builtin_convertvector(two, half2v));
        // p - hi, exact: one mixed-precision multiply-add per value where the compiler would convert
        // first.
        float2v rest;
        float r0, r1;
        asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(bits), "v"(two[0]));
        asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(bits), "v"(two[1]));
        rest[0] = r0;
        rest[1] = r1;
        h[v] = bits;
        l[v] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, half2v));
    }
    hi = __builtin_bit_cast(half8, h);
    lo = __builtin_bit_cast(half8, l);
}

/// The key, less 4 h, that accumulator r (16 a block of 32 keys) of a lane's scores belongs to.
__device__ constexpr int KeyOf(int r) { return 32 * (r / 16) + 8 * (r % 16 / 4) + r % 4; }

/// One wave owns a pair (query head, tile of 32 consecutive queries). A workgroup's four waves
/// own consecutive pairs of one kv head (the group's heads of a query tile, then the next tile's),
/// and share each step of 64 keys of K and V through LDS. Per wave and step:
///   S^T (keys x queries) = K . Q^T on the matrix cores (K the A operand from LDS, Q the B operand
///   held in registers as split planes), so a lane holds 32 keys of one query and the online
///   softmax needs only one exchange with the lane 32 away;
///   O^T (channels x queries) += V^T . P^T with P^T split into planes straight from the S^T
///   accumulators: the B operand's k slot (h, v) of lane j + 32h is key 16 s + 8 (v / 4) + 4 h +
///   v % 4 of the step, and the V^T fragment reads the same keys by two transposing LDS reads
///   (ds_read_b64_tr_b16: from 16 lanes' 8 bytes of four rows, each lane gets four keys of one
///   channel), so V lies in LDS as in the cache.
/// K and V rows go from memory to LDS without passing through registers, kStages - 1 steps ahead
/// at one barrier a step (prefill_gemm.hip has the scheme). Their 16-byte chunks are permuted by
/// the row: K's by row % 8 (eight consecutive rows read the same chunk), V's by 2 (row % 4) (a
/// transposing read takes two chunks of four rows).
///
/// What bounds it: per 64 keys and wave 64 matrix operations at head_dim 128 (32 at 64), 2048
/// (1024) cycles, and about as many of softmax instructions, of which 32 exponentials take a
/// quarter; a wave's phases follow one another, and two workgroups on a CU take twice one's time.
/// So the mask is applied only in steps that reach past a tile's first query, scores are scaled
/// inside the exponential's multiply-add, and the accumulators are rescaled only when a maximum
/// rises by 2^8 (head_dim 128: 300 vector instructions per 32 keys before, about 150 since) or by
/// the multiply-add that takes in a step's sum (64). Measured, before (one 32-key tile in LDS, V
/// transposed by hand, a barrier pair per tile) and now, us: 28 / 4 heads of 128, 777 rows after
/// 5003: 348 / 150; 2048 rows 142 / 92; 45 rows after 700: 38 / 14.6; 14 / 2 heads of 64, 613 rows
/// 28.6 / 14.9, 2048 rows 53 / 45.
///
/// Grid: kv heads fastest (an XCD then sees one or two of them), then pairs, the longest first, then
/// key chunks: whole chunks start before the tails, and an XCD does not get one chunk of every
/// tile (with the chunks before the pairs, an even number of them took a third longer). Chunk c
/// covers keys [c * C, (c + 1) * C), C = 32 * chunkTiles; a query tile with more keys than C leaves
/// each chunk's unnormalised softmax partial (running max, sum, P.V) in slot c of `part` for
/// PrefillAttnMergeKernel, one with at most C writes its planes directly.
///
/// kKeys keys (32 or 64) of a step are handled at a time. At head_dim 128 the scores and weights of
/// 64 would not fit the registers beside q and o. At 64 they do, and a wave meets half as many
/// phases; but a range that ends in the first half of a step then pays for the other half
/// (kShortTiles).
template <int kHd, int kKeys>
__global__ __launch_bounds__(kWave* kAttnWaves, 2) void PrefillAttentionKernel(
    const uint16_t* __restrict__ qhi, const uint16_t* __restrict__ qlo, const uint16_t* __restrict__ kcache,
    const uint16_t* __restrict__ vcache, uint16_t* __restrict__ ohi, uint16_t* __restrict__ olo, uint32_t rows,
    int32_t pos0, uint32_t heads, uint32_t kvHeads, uint32_t maxSeq, float scale, uint32_t chunkTiles,
    AttnPartials part)
{
    constexpr int kWaves = kAttnWaves;
    constexpr int kStages = kHd == 128 ? 2 : 3;
    // A step's products summed by themselves and added to the rescaled total: one rounding at the
    // total's size per 64 keys instead of eight, where the registers allow.
    constexpr bool kStepSums = kHd == 64;
    constexpr uint32_t kRowBytes = 2 * kHd;
    constexpr uint32_t kChunks = kHd / 8;                     // 16-byte chunks per row
    constexpr uint32_t kRowsPerLoad = kWave / kChunks;
    constexpr uint32_t kMatrixBytes = kAttnStep * kRowBytes;  // K or V of a step
    constexpr int kMatrixLoads = kMatrixBytes / 1024 / kWaves;  // per wave
    constexpr int kLoads = 2 * kMatrixLoads;
    static_assert(kWaves * kRowsPerLoad % 8 == 0, "a wave's loads share their rows' permutation");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kStages * 2 * kMatrixBytes];

    const uint32_t lane = threadIdx.x % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t h = lane / 32;
    const uint32_t group = heads / kvHeads;
    const uint32_t pairs = (rows + 31) / 32 * group;
    const uint32_t blocks = (pairs + kWaves - 1) / kWaves;
    const uint32_t kv = blockIdx.x % kvHeads;
    const uint32_t chunk = blockIdx.x / kvHeads / blocks;
    const uint32_t firstPair = (blocks - 1 - blockIdx.x / kvHeads % blocks) * kWaves;

    // The workgroup's keys: its last pair's, within the chunk. (Without any, it has no work.)
    const uint32_t lastTile = min(firstPair + kWaves - 1, pairs - 1) / group;
    const uint64_t begin = static_cast<uint64_t>(chunk) * chunkTiles * 32;
    const uint64_t last = static_cast<uint64_t>(pos0) + min(lastTile * 32 + 31, rows - 1);
    if (begin > last)
    {
        return;
    }
    const uint32_t keyBegin = static_cast<uint32_t>(begin);
    const uint32_t keyEnd = static_cast<uint32_t>(min(last + 1, begin + static_cast<uint64_t>(chunkTiles) * 32));
    const uint32_t steps = (keyEnd - keyBegin + kAttnStep - 1) / kAttnStep;

    const uint32_t pair = min(firstPair + wave, pairs - 1);
    const bool active = firstPair + wave < pairs;  // a wave past the pairs only loads
    const uint32_t qtile = pair / group;
    const uint32_t head = kv * group + pair % group;
    const uint32_t qdim = heads * kHd;
    const uint32_t m0 = qtile * 32;
    const uint32_t mq = min(m0 + lane % 32, rows - 1);
    const int32_t firstPos = pos0 + static_cast<int32_t>(m0);
    const int32_t qpos = pos0 + static_cast<int32_t>(mq);
    const int32_t lastPos = pos0 + static_cast<int32_t>(min(m0 + 31, rows - 1));

    // Load i of a wave: 1 KB of K (the first kMatrixLoads of a step) or V, rows row0, row0 + 1, ...
    // Keys past the cache reread its last row: they are masked. The addresses are a load's scalar
    // base and one of two lane offsets: more registers held for them would spill, and the wait for
    // a spilled register's return also waits for every load issued before it.
    const uint32_t ldsBase =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds));
    const uint64_t cacheBase = static_cast<uint64_t>(kv) * maxSeq * kHd;
    const uint32_t laneRow = lane / kChunks;
    const uint32_t kAt = (lane % kChunks ^ ((wave * kRowsPerLoad + laneRow) & 7u)) * 16;
    const uint32_t vLoadAt = (lane % kChunks ^ (laneRow & 3u) * 2) * 16;
    auto load = [&](uint32_t stage, uint32_t step, int i)
    {
        const bool isV = i >= kMatrixLoads;
        const uint32_t g = wave + i % kMatrixLoads * kWaves;
        const uint32_t row0 = min(keyBegin + step * kAttnStep + g * kRowsPerLoad, maxSeq - 1);
        const uint16_t* base = (isV ? vcache : kcache) + cacheBase + static_cast<uint64_t>(row0) * kHd;
        const uint32_t offset = min(laneRow, maxSeq - 1 - row0) * kRowBytes + (isV ? vLoadAt : kAt);
        LoadToLds(ldsBase + stage * 2 * kMatrixBytes + wave * 1024,
                  isV * kMatrixBytes + i % kMatrixLoads * kWaves * 1024, offset, base);
    };

    // Scores are scaled by |scale| (in log2 units) inside the exponential, so that the running
    // maximum can be of the raw scores; a negative scale turns q's sign, and 0 clears q.
    half8 qh[kHd / 16], ql[kHd / 16];
    {
        const uint64_t at = static_cast<uint64_t>(mq) * qdim + head * kHd + 8 * h;
#pragma unroll
        for (int s = 0; s < kHd / 16; ++s)
        {
            qh[s] = *reinterpret_cast<const half8*>(qhi + at + 16 * s);
            ql[s] = *reinterpret_cast<const half8*>(qlo + at + 16 * s);
        }
        if (scale <= 0.0f)
        {
            const _Float16 sign = static_cast<_Float16>(scale < 0.0f ? -1.0f : 0.0f);
#pragma unroll
            for (int s = 0; s < kHd / 16; ++s)
            {
                qh[s] *= sign;
                ql[s] *= sign;
            }
        }
    }
    const float scaleLog2 = scale == 0.0f ? 1.0f : fabsf(scale) * 1.44269504088896340736f;
#pragma unroll
    for (uint32_t s = 0; s < kStages - 1; ++s)
    {
        if (s < steps)
        {
#pragma unroll
            for (int i = 0; i < kLoads; ++i)
            {
                load(s, s, i);
            }
        }
    }

    // q's arrival is waited for here, outside the loop: the compiler's own wait would also cover the
    // loads it does not see, in every step.
#pragma unroll
    for (int s = 0; s < kHd / 16; ++s)
    {
        asm volatile("" : "+v"(qh[s]), "+v"(ql[s]));
    }

    floatx16 o[kHd / 32];
#pragma unroll
    for (int c = 0; c < kHd / 32; ++c)
    {
        o[c] = floatx16{};
    }
    float runMax = -INFINITY;  // of the raw scores
    float shift = 0.0f;        // runMax scaled, in log2 units
    float runSum = 0.0f;
    const uint32_t kRow = lane % 32;
    const uint32_t vRow = 4 * h + lane % 16 / 4;
    const uint32_t vChunk = (lane / 16 % 2 * 2 + lane % 4 / 2) ^ (vRow & 3u) * 2;
    const uint32_t vAt = vRow * kRowBytes + lane % 2 * 8;

    uint32_t stage = 0;
    for (uint32_t t = 0; t < steps; ++t, stage = stage + 1 == kStages ? 0 : stage + 1)
    {
        const uint32_t ahead = min(static_cast<uint32_t>(kStages - 2), steps - 1 - t);
        if (kStages <= 2 || ahead == 0)
        {
            WaitAndMeet<0>();
        }
        else
        {
            WaitAndMeet<kLoads>();
        }
        if (t + kStages - 1 < steps)
        {
            const uint32_t freed = stage == 0 ? kStages - 1 : stage - 1;
#pragma unroll
            for (int i = 0; i < kLoads; ++i)
            {
                load(freed, t + kStages - 1, i);
            }
        }
        if (!active)
        {
            continue;
        }
#pragma unroll 1
        for (uint32_t first = 0; first < kAttnStep; first += kKeys)
        {
            const int32_t key0 = static_cast<int32_t>(keyBegin + t * kAttnStep + first);
            if (key0 > lastPos)
            {
                break;
            }
            const uint8_t* kTile = lds + (stage * 2 * kMatrixBytes + first * kRowBytes);
            const uint8_t* vTile = kTile + kMatrixBytes;
            floatx16 st[kKeys / 32], low[kKeys / 32];  // two sums: independent operations in a row
#pragma unroll
            for (int b = 0; b < kKeys / 32; ++b)
            {
                st[b] = floatx16{};
                low[b] = floatx16{};
            }
#pragma unroll
            for (int s = 0; s < kHd / 16; ++s)
            {
                half8 kf[kKeys / 32];
#pragma unroll
                for (int b = 0; b < kKeys / 32; ++b)
                {
                    kf[b] = *reinterpret_cast<const half8*>(kTile + (32 * b + kRow) * kRowBytes +
                                                            ((2 * s + h) ^ (kRow & 7u)) * 16);
                    st[b] = Mfma(kf[b], qh[s], st[b]);
                }
#pragma unroll
                for (int b = 0; b < kKeys / 32; ++b)
                {
                    low[b] = Mfma(kf[b], ql[s], low[b]);
                }
            }
#pragma unroll
            for (int b = 0; b < kKeys / 32; ++b)
            {
                st[b] += low[b];
            }
            // Keys that a query does not see (KeyOf) score -inf: weight 0.
            if (key0 + kKeys - 1 > firstPos)
            {
                int32_t visible = qpos - key0 - 4 * static_cast<int32_t>(h);
                asm volatile("" : "+v"(visible));  // a branch, not selects in every step
#pragma unroll
                for (int r = 0; r < kKeys / 2; ++r)
                {
                    // By a mask in a vector register: compares would hold a scalar pair each.
                    const uint32_t hidden = static_cast<uint32_t>((visible - KeyOf(r)) >> 31);
                    const uint32_t score = __float_as_uint(st[r / 16][r % 16]);
                    st[r / 16][r % 16] = __uint_as_float((hidden & 0xFF800000u) | (~hidden & score));
                }
            }
            float tileMax = -INFINITY;
#pragma unroll
            for (int r = 0; r < kKeys / 2; ++r)
            {
                tileMax = fmaxf(tileMax, st[r / 16][r % 16]);
            }
            tileMax = fmaxf(tileMax, PartnerLane<32>(tileMax));
            // A chunk of a split tile may hold no key of a query yet: its maximum stays -inf, and
            // every weight is 0 by the mask.
            //
            // Weights are relative to `shift`, which follows the (scaled, rounded) maximum only once
            // that is 2^8 past it: weights up to 256 keep the planes' relative precision (f16 ends
            // at 65504), and rescaling the accumulators, which some query of the tile would need
            // in most steps, becomes rare.
            const float top = tileMax * scaleLog2;
            const bool rises = tileMax != -INFINITY && (runMax == -INFINITY || top > shift + 8.0f);
            float factor = 1.0f;
            if (__any(rises))
            {
                const float newShift = rises ? top : shift;
                factor = rises ? (runMax == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(shift - newShift)) : 1.0f;
                runMax = rises ? tileMax : runMax;
                shift = newShift;
                if constexpr (!kStepSums)
                {
#pragma unroll
                    for (int c = 0; c < kHd / 32; ++c)
                    {
                        o[c] *= factor;
                    }
                }
            }
            float p[kKeys / 2];
#pragma unroll
            for (int r = 0; r < kKeys / 2; ++r)
            {
                p[r] = __builtin_amdgcn_exp2f(fmaf(st[r / 16][r % 16], scaleLog2, -shift));
            }
            float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < kKeys / 2; ++r)
            {
                sum[r % 4] += p[r];
            }
            runSum = fmaf(runSum, factor, (sum[0] + sum[1]) + (sum[2] + sum[3]));
            half8 ph[kKeys / 16], pl[kKeys / 16];
#pragma unroll
            for (int s = 0; s < kKeys / 16; ++s)
            {
                SplitWeights(p + 8 * s, ph[s], pl[s]);
            }
            // Rows past the tile's last query position may hold anything (NaN, inf): their weight
            // is 0, and 0 * NaN would poison every query of the tile, so they enter as zeros. Word w
            // of step s holds keys 16 s + 8 (w / 2) + 4 h + 2 (w % 2) and the next. (Masked in every
            // step: a second copy of the products for the last one would move the accumulators
            // about.)
            uint32_t keep[kKeys / 4];
#pragma unroll
            for (int w = 0; w < kKeys / 4; ++w)
            {
                keep[w] = 0xFFFFFFFFu;
            }
            if (key0 + kKeys - 1 > lastPos)
            {
                int32_t left = lastPos - key0 - 4 * static_cast<int32_t>(h);
                asm volatile("" : "+v"(left));
#pragma unroll
                for (int w = 0; w < kKeys / 4; ++w)
                {
                    const int key = 8 * (w / 2) + 2 * (w % 2);
                    const uint32_t past0 = static_cast<uint32_t>((left - key) >> 31);
                    const uint32_t past1 = static_cast<uint32_t>((left - key - 1) >> 31);
                    keep[w] = ~((past0 & 0xFFFFu) | (past1 & 0xFFFF0000u));
                }
            }
#pragma unroll
            for (int c = 0; c < kHd / 32; ++c)
            {
                floatx16 add = kStepSums ? floatx16{} : o[c];
#pragma unroll
                for (int s = 0; s < kKeys / 16; ++s)
                {
                    uint4v bits;
#pragma unroll
                    for (int half = 0; half < 2; ++half)
                    {
                        const uint8_t* from = vTile + vAt + (16 * s + 8 * half) * kRowBytes + (vChunk ^ (4u * c)) * 16;
                        const uint2v four = __builtin_bit_cast(
                            uint2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                        (__attribute__((address_space(3))) short4v*)(const_cast<uint8_t*>(from))));
                        bits[2 * half] = four[0] & keep[4 * s + 2 * half];
                        bits[2 * half + 1] = four[1] & keep[4 * s + 2 * half + 1];
                    }
                    const half8 vf = __builtin_bit_cast(half8, bits);
                    add = Mfma(vf, ph[s], add);
                    add = Mfma(vf, pl[s], add);
                }
                if constexpr (kStepSums)
                {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                    {
                        o[c][r] = fmaf(o[c][r], factor, add[r]);
                    }
                }
                else
                {
                    o[c] = add;
                }
            }
        }
    }

    const float total = runSum + PartnerLane<32>(runSum);
    const uint32_t m = m0 + lane % 32;
    if (!active || m >= rows || keyBegin > static_cast<uint32_t>(lastPos))
    {
        return;
    }
    if (AttnKeyTiles(qtile, rows, pos0) > chunkTiles)
    {
        // Slot `chunk`: the running max and sum of the query (both halves of the wave agree on
        // the max; their sums are added), and its unnormalised P.V.
        const uint64_t at = (static_cast<uint64_t>(chunk) * rows + m) * heads + head;
        if (h == 0)
        {
            part.max[at] = runMax == -INFINITY ? -INFINITY : shift;
            part.sum[at] = total;
        }
#pragma unroll
        for (int c = 0; c < kHd / 32; ++c)
        {
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                const uint32_t channel = c * 32 + 8 * q + 4 * h;
                *reinterpret_cast<float4*>(part.acc + at * kHd + channel) =
                    make_float4(o[c][4 * q], o[c][4 * q + 1], o[c][4 * q + 2], o[c][4 * q + 3]);
            }
        }
        return;
    }
    const float inv = 1.0f / total;
    const uint64_t base = static_cast<uint64_t>(m) * qdim + head * kHd;
#pragma unroll
    for (int c = 0; c < kHd / 32; ++c)
    {
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            const uint32_t channel = c * 32 + 8 * q + 4 * h;
            StoreSplit4(ohi, olo, base + channel, o[c][4 * q] * inv, o[c][4 * q + 1] * inv, o[c][4 * q + 2] * inv,
                        o[c][4 * q + 3] * inv);
        }
    }
}

/// Key chunks and a chunk's length (in tiles of 32 keys) of one launch.
struct AttnPlan
{
    uint32_t chunks, chunkTiles;
};

/// The fewest estimated us: the workgroups' steps over 256 CUs and half of the longest one at the
/// end, or the longest one alone; with chunks, the partials' way to memory and back and the merge.
/// A CU takes 2.2 us per step of a workgroup (head_dim 64: 1.5), whether it holds one or two. Over
/// 17 measured launches (20 to 2048 rows at cache rows 0 to 5000, both head sizes) the choice was
/// within 8 % of the fastest. The merge of a few rows at head_dim 64 costs less (32 rows at cache row
/// 100, 14 / 2 heads, three steps in one chunk 9.6 us, in three 8.5; 250 rows at row 0, four steps,
/// 10.8 / 10.0).
///
/// At head_dim 128, whose sums run over a whole chunk (kStepSums), a chunk is at most twice an
/// eighth of the range or 1024 keys: the error against 64 bits stays that of eighths and 512 keys
/// with the scores' two planes in one sum (8.6e-7 at 5780 keys, 7.4e-7 at 5048). At 64 one chunk may
/// hold everything (80 rows at cache row 0, 14 / 2 heads: 6.8 us in one chunk, 9.0 in two).
AttnPlan PlanAttention(uint32_t rows, int32_t pos0, uint32_t heads, uint32_t kvHeads, uint32_t headDim, bool split)
{
    const uint32_t tiles = CeilDiv(rows, 32);
    const uint32_t longest = AttnKeyTiles(tiles - 1, rows, pos0);
    const double stepUs = headDim == 128 ? 2.2 : 1.5;
    const double blocks = static_cast<double>(CeilDiv(static_cast<uint64_t>(tiles) * (heads / kvHeads), kAttnWaves)) * kvHeads;
    const double range = (AttnKeyTiles(0, rows, pos0) + longest) / 2.0;  // key tiles of the average workgroup
    const uint32_t whole = CeilDiv(longest, 2) * 2;
    const uint32_t cap = headDim == 128 ? 2 * std::max(16u, CeilDiv(longest, 8)) : whole;
    AttnPlan best{1, whole};
    double bestUs = std::numeric_limits<double>::infinity();
    for (uint32_t chunks = 1; chunks <= (split ? kAttnMaxChunks : 1); ++chunks)
    {
        const uint32_t chunkTiles = CeilDiv(CeilDiv(longest, chunks), 2) * 2;  // whole steps
        if (CeilDiv(longest, chunkTiles) != chunks || (split && chunkTiles > cap && chunks < kAttnMaxChunks))
        {
            continue;
        }
        const double all = blocks * range / 2.0 * stepUs / 256.0;
        const double one = chunkTiles / 2 * stepUs;
        double us = std::max(all + one / 2.0, one + 3.0);
        if (chunks > 1)
        {
            // (A small merge follows at once; one of a megabyte or more starts with its own loads.)
            const double partialsUs = (range / chunkTiles) * rows * heads * (headDim + 2) * 4.0 / 5.0e6;
            us += 2.0 * partialsUs + (headDim == 128 ? 4.0 : 2.35 + std::min(2.75 * partialsUs, 1.65));
        }
        if (us < bestUs)
        {
            bestUs = us;
            best = AttnPlan{chunks, chunkTiles};
        }
    }
    return best;
}
/// At head_dim 64, ranges of up to this many tiles of 32 keys are handled 32 keys at a time. 14 / 2
/// heads, us, 64 keys / 32: one row at cache row 0 4.8 / 4.0, 32 rows 6.3 / 5.4, 64 rows 6.3 / 6.2.
/// (Up to six tiles 32 keys are as fast or faster, 80 rows 6.8 / 6.3; but the sums meet the total
/// twice as often, and one row after 100 is 2.1e-7 / 2.5e-7 off its 64-bit value.)
constexpr uint32_t kShortTiles = 2;

uint32_t KeysAtATime(uint32_t rows, int32_t pos0, uint32_t headDim)
{
    return headDim == 64 && AttnKeyTiles(CeilDiv(rows, 32) - 1, rows, pos0) > kShortTiles ? 64 : 32;
}
}  // namespace

hipError_t LaunchPrefillAttention(hipStream_t s, const uint16_t* qhi, const uint16_t* qlo, const uint16_t* kcache,
                                  const uint16_t* vcache, uint16_t* ohi, uint16_t* olo, uint32_t rows, int32_t pos0,
                                  uint32_t heads, uint32_t kvHeads, uint32_t headDim, uint32_t maxSeq, float scale,
                                  float* workspace, size_t workspaceFloats)
{
    if (rows == 0 || kvHeads == 0 || heads % kvHeads != 0 || heads / kvHeads > 8 || pos0 < 0 ||
        static_cast<uint64_t>(pos0) + rows > maxSeq || (headDim != 64 && headDim != 128))
    {
        return hipErrorInvalidValue;
    }
    const bool split =
        workspace != nullptr && workspaceFloats >= PrefillAttentionWorkspaceFloats(rows, heads, headDim);
    const AttnPlan plan = PlanAttention(rows, pos0, heads, kvHeads, headDim, split);
    AttnPartials part{};
    if (plan.chunks > 1)
    {
        const size_t stats = static_cast<size_t>(kAttnMaxChunks) * rows * heads;
        part = AttnPartials{workspace, workspace + stats, workspace + 2 * stats};
    }
    const uint32_t pairs = CeilDiv(rows, 32) * (heads / kvHeads);
    const dim3 grid(CeilDiv(pairs, kAttnWaves) * plan.chunks * kvHeads);
    const auto kernel = headDim == 128                          ? PrefillAttentionKernel<128, 32>
                        : KeysAtATime(rows, pos0, headDim) == 32 ? PrefillAttentionKernel<64, 32>
                                                                 : PrefillAttentionKernel<64, 64>;
    hipLaunchKernelGGL(kernel, grid, dim3(kWave * kAttnWaves), 0, s, qhi, qlo, kcache, vcache, ohi, olo, rows, pos0,
                       heads, kvHeads, maxSeq, scale, plan.chunkTiles, part);
    if (plan.chunks > 1)
    {
        const uint64_t threads = static_cast<uint64_t>(rows) * heads * (headDim / 4);
        hipLaunchKernelGGL(PrefillAttnMergeKernel, dim3(static_cast<uint32_t>(CeilDiv(threads, 256))), dim3(256), 0, s,
                           part, ohi, olo, rows, pos0, heads, headDim, plan.chunkTiles);
    }
    return hipGetLastError();
}
}  // namespace muyo

// For the tests (no device needed): the chunks of a launch, their length in tiles of 32 keys, and the
// keys handled at a time.
extern "C" void muyo_prefill_attention_plan(uint32_t rows, int32_t pos0, uint32_t heads, uint32_t kvHeads,
                                            uint32_t headDim, uint32_t workspace, uint32_t plan[3])
{
    const muyo::AttnPlan p = muyo::PlanAttention(rows, pos0, heads, kvHeads, headDim, workspace != 0);
    plan[0] = p.chunks;
    plan[1] = p.chunkTiles;
    plan[2] = muyo::KeysAtATime(rows, pos0, headDim);
}
