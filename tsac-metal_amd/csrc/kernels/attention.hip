// Causal multi-head attention with the reference's exact arithmetic
// (src/scalar/attention.cpp:12-131):
//   * scores: one serial fma chain over the head coordinates (ascending), times scale;
//   * keys in 64-position blocks: block max, original_exp(score - max), pair-tree
//     block sum, per-coordinate serial fma value sums (BF16-rounded when the
//     query's history exceeds 64 positions or during replay);
//   * blocks merged in ascending order with the online-softmax recurrence.
// Matrix cores would reorder those sums, so everything runs on the VALU.
//
// Decode (one query per sequence): each (sequence, head)'s 64-key blocks are
// spread over several workgroups of one launch, one wave per block; the last
// workgroup to arrive merges the block records in ascending order.
// Prefill (encode, all queries known): one workgroup per (sequence, head, query
// tile), one wave per causal key block, the blocks' sums merged in ascending order.
#include "attention.hpp"
#include "device_numeric.hpp"

namespace tsac_hip
{
namespace
{
__device__ __forceinline__ void rotate_pair(float& re, float& im, const uint16_t* c)
{
    const float cosine = bf16_to_float(c[0]), sine = bf16_to_float(c[1]);
    const float im_sine = im * sine;
    const float re_sine = re * sine;
    const float r = __builtin_fmaf(re, cosine, -im_sine);
    const float i = __builtin_fmaf(im, cosine, re_sine);
    re = round_bf16(r);
    im = round_bf16(i);
}

// ------------------------------------------------------------------ decode

// Splits each row's Q, K and V out of the projection output, applies rotary to
// Q and K when a table is given, appends K and V to the caches at `position`.
__global__ void append_kernel(const uint16_t* __restrict__ qkv, int rows, int width, int head_width,
                              const uint16_t* __restrict__ rotation, uint16_t* __restrict__ query,
                              uint16_t* keys, uint16_t* values, std::size_t row_stride)
{
    const int pairs = width / 2;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows * pairs;
         i += gridDim.x * blockDim.x)
    {
        const int row = i / pairs, j = 2 * (i % pairs);
        const uint16_t* src = qkv + std::size_t(row) * 3 * width;
        float qr = bf16_to_float(src[j]), qi = bf16_to_float(src[j + 1]);
        float kr = bf16_to_float(src[width + j]), ki = bf16_to_float(src[width + j + 1]);
        if (rotation)
        {
            const uint16_t* c = rotation + j % head_width;
            rotate_pair(qr, qi, c);
            rotate_pair(kr, ki, c);
        }
        query[std::size_t(row) * width + j] = float_to_bf16(qr);
        query[std::size_t(row) * width + j + 1] = float_to_bf16(qi);
        uint16_t* k = keys + std::size_t(row) * row_stride;
        uint16_t* v = values + std::size_t(row) * row_stride;
        k[j] = float_to_bf16(kr);
        k[j + 1] = float_to_bf16(ki);
        v[j] = src[2 * width + j];
        v[j + 1] = src[2 * width + j + 1];
    }
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Waves per decode workgroup; each wave computes one 64-key block's record.
constexpr int decode_waves = 4;


// Workgroups per (sequence, head) for a history of `blocks` key blocks.
constexpr int decode_splits(int blocks)
{
    return (blocks + decode_waves - 1) / decode_waves;
}

// One query per (sequence, head) over its `time` cached keys, split over
// decode_splits(blocks) workgroups of decode_waves waves: wave w of split s
// computes the record [max, block sum, value sums[HW]] of block
// s * decode_waves + w. With one split the records stay in LDS; otherwise
// they go to `partial` ([sequence * heads + head][blocks][2 + HW]) and each
// workgroup counts its arrival in `arrivals[sequence * heads + head]` (zero
// on entry, zero again on exit): the last to arrive copies every record into
// LDS and merges them in ascending block order, so the counter only hands
// the merge over and the summation order is the single-workgroup one.
//
// A block's key and value rows are read whole (16 bytes per lane, so a load
// covers 64 / (HW / 8) rows) and pass through LDS: each lane takes its key
// row, then its value column.
//
// The merge's running maxima are a scan with the recurrence's own update
// (keep the running maximum unless it is smaller: the first of equal values
// wins), which is associative without NaNs, so every block's factors come at
// once and only the two-operation total/numerator recurrence stays
// sequential; with a NaN maximum the merge runs the plain loop.
template <int HW>
__global__ __launch_bounds__(decode_waves * 64) void decode_attention_kernel(
    const uint16_t* __restrict__ query, const uint16_t* __restrict__ keys,
    const uint16_t* __restrict__ values, std::size_t sequence_stride, int width, int time,
    int heads, float scale, int round_values, float* __restrict__ partial, unsigned* __restrict__ arrivals,
    uint16_t* __restrict__ out)
{
    constexpr int chunks = HW / 8;            // 16-byte chunks per row
    constexpr int rows_per_load = 64 / chunks;
    extern __shared__ float records[];        // [blocks][2 + HW]
    __shared__ uint4 staged[decode_waves][64 * chunks]; // each wave's key rows, then value rows
    __shared__ float weights[decode_waves][64];
    __shared__ float4 factors[64]; // the merge's per-block (old scale, new scale, block sum)
    __shared__ int merging;
    const int blocks = (time + 63) / 64;
    const int splits = decode_splits(blocks);
    const int pair = blockIdx.x / splits, split = blockIdx.x % splits;
    const int sequence = pair / heads, head = pair % heads;
    const int lane = threadIdx.x % wave, warp = __builtin_amdgcn_readfirstlane(int(threadIdx.x / wave));
    const uint16_t* k = keys + std::size_t(sequence) * sequence_stride + head * HW;
    const uint16_t* v = values + std::size_t(sequence) * sequence_stride + head * HW;
    // Lane l sums value column l (HW = 64) or columns 2l and 2l + 1 (HW = 128).
    constexpr int per_lane = HW / 64;
    float* const shared_records = partial + std::size_t(pair) * blocks * (2 + HW);
    const int block = split * decode_waves + warp;
    if (block < blocks)
    {
        const int start = block * 64;
        const int count = time - start < 64 ? time - start : 64;
        // The block's key rows and value rows, whole rows at a time (16 bytes
        // per lane, so a load covers 64 / (HW / 8) rows), all requested
        // before any is used. Rows past the history lie beyond the buffers'
        // ends and read zero; their scores are dropped and their values not
        // used. The row offset goes in the range-checked vector offset (the
        // scalar offset is not checked).
        const __amdgpu_buffer_rsrc_t key_rows =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(k), 0, time * width * 2, 0x00020000);
        const __amdgpu_buffer_rsrc_t value_rows =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(v), 0, time * width * 2, 0x00020000);
        const int lane_offset = (lane / chunks) * width * 2 + (lane % chunks) * 16;
        uint4 key_data[chunks], rows[chunks];
#pragma unroll
        for (int i = 0; i < chunks; ++i)
        {
            const u32x4 r = __builtin_amdgcn_raw_buffer_load_b128(
                key_rows, lane_offset + (start + i * rows_per_load) * width * 2, 0, 0);
            key_data[i] = make_uint4(r.x, r.y, r.z, r.w);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < chunks; ++i)
        {
            const u32x4 r = __builtin_amdgcn_raw_buffer_load_b128(
                value_rows, lane_offset + (start + i * rows_per_load) * width * 2, 0, 0);
            rows[i] = make_uint4(r.x, r.y, r.z, r.w);
        }
        __builtin_amdgcn_sched_barrier(0); // every load issued before the first wait
        // Keys through LDS to one row per lane; chunk c of row r is kept at
        // r * chunks + (c ^ (r % 8)), so neither the row-wise writes nor the
        // lane-per-row reads meet in a bank.
#pragma unroll
        for (int i = 0; i < chunks; ++i)
        {
            const int r = i * rows_per_load + lane / chunks, c = lane % chunks;
            staged[warp][r * chunks + (c ^ (r & 7))] = key_data[i];
        }
        __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
        __builtin_amdgcn_wave_barrier();
        uint4 key[chunks];
#pragma unroll
        for (int c = 0; c < chunks; ++c)
        {
            key[c] = staged[warp][lane * chunks + (c ^ (lane & 7))];
        }
        // The query, uniform over the workgroup, in scalar registers.
        const uint32_t* q = reinterpret_cast<const uint32_t*>(query + std::size_t(sequence) * width + head * HW);
        float dot = 0.0f;
#pragma unroll
        for (int c = 0; c < chunks; ++c)
        {
            const uint4 u = key[c];
            const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const uint32_t pair_q = __builtin_amdgcn_readfirstlane(q[4 * c + i]);
                dot = __builtin_fmaf(__uint_as_float(pair_q << 16), __uint_as_float(w[i] << 16), dot);
                dot = __builtin_fmaf(__uint_as_float(pair_q & 0xffff0000u), __uint_as_float(w[i] & 0xffff0000u), dot);
            }
        }
        const float score = lane < count ? dot * scale : -__builtin_inff();
        const float maximum = group_max<wave>(score);
        float e = 0.0f;
        if (lane < count)
        {
            e = original_exp(score - maximum);
        }
        const float sum = tree_sum<wave>(e);
        weights[warp][lane] = e;
#pragma unroll
        for (int i = 0; i < chunks; ++i)
        {
            staged[warp][i * 64 + lane] = rows[i];
        }
        __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0): the wave's weights and values are in
        __builtin_amdgcn_wave_barrier();
        const uint16_t* column16 = reinterpret_cast<const uint16_t*>(staged[warp]) + lane;
        const uint32_t* column32 = reinterpret_cast<const uint32_t*>(staged[warp]) + lane;
        float s0 = 0.0f, s1 = 0.0f;
        const auto accumulate = [&](int t)
        {
            const float w = weights[warp][t];
            if constexpr (per_lane == 2)
            {
                const uint32_t p = column32[t * 64];
                s0 = __builtin_fmaf(__uint_as_float(p << 16), w, s0);
                s1 = __builtin_fmaf(__uint_as_float(p & 0xffff0000u), w, s1);
            }
            else
            {
                s0 = __builtin_fmaf(__uint_as_float(uint32_t(column16[t * 64]) << 16), w, s0);
            }
        };
        if (count == 64)
        {
#pragma unroll
            for (int t = 0; t < 64; ++t)
            {
                accumulate(t);
            }
        }
        else
        {
            for (int t = 0; t < count; ++t)
            {
                accumulate(t);
            }
        }
        const std::size_t at = std::size_t(block) * (2 + HW);
        // Records for the merge of another workgroup go out as device-coherent
        // stores, so no cache needs writing back before the arrival is counted.
        const auto put = [&](int i, float value)
        {
            if (splits == 1)
            {
                records[at + i] = value;
            }
            else
            {
                __hip_atomic_store(shared_records + at + i, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        };
        if (lane == 0)
        {
            put(0, maximum);
            put(1, sum);
        }
        put(2 + per_lane * lane, round_values ? round_bf16(s0) : s0);
        if constexpr (per_lane == 2)
        {
            put(3 + per_lane * lane, round_values ? round_bf16(s1) : s1);
        }
    }
    if (splits > 1)
    {
        // Every wave's records are written before the workgroup counts its
        // arrival; the last to arrive resets the counter and merges.
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (threadIdx.x == 0)
        {
            const unsigned before =
                __hip_atomic_fetch_add(arrivals + pair, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            merging = before == unsigned(splits - 1);
            if (merging)
            {
                __hip_atomic_store(arrivals + pair, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();
        if (!merging)
        {
            return;
        }
    }
    else
    {
        __syncthreads();
    }
    if (warp != 0)
    {
        return;
    }
    // Ordered merge (src/scalar/attention.cpp:86-101) by one wave, over
    // chunks of 64 blocks: lane b holds block b's maximum and sum, every lane
    // its value sums of all 64 blocks (read from LDS with one split, with
    // device-coherent loads from `partial` otherwise, all requested at once).
    const auto scales_of = [](float running, float maximum, float& old_scale, float& new_scale)
    {
        const float factor = original_exp(-__builtin_fabsf(maximum - running));
        old_scale = running > maximum ? 1.0f : factor;
        new_scale = running > maximum ? factor : 1.0f;
    };
    float numerator[per_lane];
#pragma unroll
    for (int c = 0; c < per_lane; ++c)
    {
        numerator[c] = 0.0f;
    }
    float total = 0.0f;
    float carry = -__builtin_inff();
    for (int chunk = 0; chunk < blocks; chunk += wave)
    {
        const int here = blocks - chunk < wave ? blocks - chunk : wave;
        const bool live = lane < here;
        // Straight-line loads in groups of eight blocks, every one requested
        // before the first is waited for. A group may read up to seven
        // records past the last block (the records are followed by that much
        // padding); those values are replaced below.
        float first[2];
        float column[wave][per_lane];
        const auto gather = [&](auto load)
        {
            const int b = chunk + (live ? lane : here - 1);
            first[0] = load(std::size_t(b) * (2 + HW));
            first[1] = load(std::size_t(b) * (2 + HW) + 1);
            const std::size_t base = std::size_t(chunk) * (2 + HW) + 2 + per_lane * lane;
#pragma unroll
            for (int g = 0; g < wave / 8; ++g)
            {
                if (g * 8 < here)
                {
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                    {
#pragma unroll
                        for (int c = 0; c < per_lane; ++c)
                        {
                            column[g * 8 + j][c] = load(base + std::size_t(g * 8 + j) * (2 + HW) + c);
                        }
                    }
                }
            }
        };
        if (splits == 1)
        {
            gather([&](std::size_t at) { return records[at]; });
        }
        else
        {
            gather([&](std::size_t at)
                   { return __hip_atomic_load(shared_records + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); });
        }
        // Lanes past the last block step with old scale 1, new scale 0 and
        // sums of -0, which leave the total and numerators exactly as they
        // are, so the steps need no per-block branch.
        const float maximum = live ? first[0] : -__builtin_inff();
        const float block_sum = live ? first[1] : -0.0f;
        float old_scale = 1.0f, new_scale = 0.0f;
        if (__any(__builtin_isnan(maximum)))
        {
            // The plain running maximum, one block at a time.
            float running = carry;
            for (int i = 0; i < here; ++i)
            {
                const float m = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(maximum), i));
                float o, n;
                scales_of(running, m, o, n);
                if (lane == i)
                {
                    old_scale = o;
                    new_scale = n;
                }
                running = running < m ? m : running;
            }
            carry = running;
        }
        else
        {
            const float scanned = running_max_scan(maximum);
            const float inclusive = carry < scanned ? scanned : carry;
            scales_of(previous_lane(inclusive, carry), maximum, old_scale, new_scale);
            carry = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inclusive), here - 1));
        }
        // Each block's factors go through LDS, so the steps read them as
        // operands (one broadcast read per block) instead of moving them lane
        // by lane into scalar registers.
        factors[lane] = make_float4(live ? old_scale : 1.0f, live ? new_scale : 0.0f, block_sum, 0.0f);
        __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int g = 0; g < wave / 8; ++g)
        {
            if (g * 8 < here)
            {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                {
                    const float4 f = factors[g * 8 + j];
                    total = __builtin_fmaf(f.z, f.y, total * f.x);
#pragma unroll
                    for (int c = 0; c < per_lane; ++c)
                    {
                        const float sum = g * 8 + j < here ? column[g * 8 + j][c] : -0.0f;
                        numerator[c] = __builtin_fmaf(sum, f.y, numerator[c] * f.x);
                    }
                }
            }
        }
        __builtin_amdgcn_wave_barrier(); // the factors are read before the next chunk's are written
    }
    const float reciprocal = 1.0f / total;
    uint16_t* o = out + std::size_t(sequence) * width + head * HW + per_lane * lane;
    if constexpr (per_lane == 2)
    {
        *reinterpret_cast<uint32_t*>(o) =
            float_to_bf16(numerator[0] * reciprocal) | (uint32_t(float_to_bf16(numerator[1] * reciprocal)) << 16);
    }
    else
    {
        *o = float_to_bf16(numerator[0] * reciprocal);
    }
}


// ------------------------------------------------------------------ prefill

constexpr int tile = 64; // keys of a block
constexpr unsigned grid_reach = 65535; // query tiles along y; z takes those past it

// 16 bytes at any 2-byte-aligned address.
__device__ __forceinline__ u32x4 load16(const uint16_t* from)
{
    u32x4 u;
    __builtin_memcpy(&u, from, 16);
    return u;
}

// Rotary (optional) of eight consecutive values.
__device__ __forceinline__ u32x4 rotate8(u32x4 u, u32x4 coefficients)
{
#pragma unroll
    for (int p = 0; p < 4; ++p)
    {
        float re = bf16_to_float(uint16_t(u[p] & 0xffff));
        float im = bf16_to_float(uint16_t(u[p] >> 16));
        const uint16_t pair[2] = {uint16_t(coefficients[p] & 0xffff), uint16_t(coefficients[p] >> 16)};
        rotate_pair(re, im, pair);
        u[p] = float_to_bf16(re) | (uint32_t(float_to_bf16(im)) << 16);
    }
    return u;
}

__device__ __forceinline__ void widen8(u32x4 u, float (&v)[8])
{
#pragma unroll
    for (int p = 0; p < 4; ++p)
    {
        v[2 * p] = __uint_as_float(u[p] << 16);
        v[2 * p + 1] = __uint_as_float(u[p] & 0xffff0000u);
    }
}

// One wave's LDS accesses are served in order; this keeps the compiler from
// moving them across a change of a wave's own tile.
__device__ __forceinline__ void tile_fence()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// LDS of a workgroup of W waves: the query tile, each wave's key (32
// coordinates of 64 keys at a time), weight (16 keys x the queries, in the keys'
// place) and value tiles (16 keys x 64 coordinates), and the merged state that
// the waves hand on block by block. Rows are padded so that eight lanes reading or
// writing 16 bytes of eight rows meet eight different 16-byte banks.
constexpr int phase_coordinates = 32, chunk_keys = 16, value_coordinates = 64;

template <int HW, int W, int queries> struct PrefillShared
{
    static constexpr int per_lane = queries / 8;
    static constexpr int q_row = HW + 8, k_row = phase_coordinates + 8, p_row = queries + 4;
    union Wave
    {
        uint16_t k[tile * k_row];
        struct
        {
            float p[chunk_keys * p_row];
            uint16_t v[chunk_keys * value_coordinates];
        };
    };
    alignas(16) uint16_t q[queries * q_row];
    alignas(16) Wave wave[W];
    alignas(16) f32x4 numerator[HW / 64 * per_lane * 2][64]; // per lane: the lane's own sums
    float maximum[queries], total[queries];
    int turn[HW / value_coordinates];
};

// A workgroup takes 8, 16 or 32 queries of one (sequence, head); its W waves take the
// causal 64-key blocks in turn, each whole: lane (lq, lk) = (lane / 8, lane % 8)
// holds queries lq + 8 a and, for scores, keys lk + 8 b, so that the 8-lane
// butterfly on each register followed by the register pair tree is exactly the
// balanced pair tree over the block's 64 positions; for value sums it holds eight
// coordinates of the same queries. The block's sums join the running state in
// ascending block order: a wave waits for its block's turn, which the wave of the
// block before passes on, so the first block's wave never waits and every wait ends.
//
// Bound by the issue of the waves that are resident: the chains over coordinates and
// keys leave no room for matrix instructions, and a wave issues one VALU instruction per
// 4 cycles at most (two waves of a SIMD issue side by side: 59-70 T fma/s for the whole
// chip on register operands). Counters of 3 sequences of 861 rows, 16 heads of 64 (4 x 32):
// 7,500 VALU instructions a block, 4,096 of them the chains' fmas, in 50 k cycles; a wave
// issues one in 60% of its 4-cycle slots and waits for memory or LDS in 21%, and a
// SIMD holds 1.45 waves on average, so that the launch reaches 44% of what two waves a SIMD
// issue. A block's time makes the longest query tile's rounds the floor of a short launch.
// Tiles of 64 queries (8 x 8 sums a lane, 13% fewer instructions) made those rounds twice
// as long: 160 us against 136. Four waves per SIMD (128 registers) spill and gain nothing.
// One workgroup walking a tile's blocks one after the other with 4 x 4 sums a thread
// (before) was bound by its LDS reads and barriers. us by events around repeated
// launches, rotated, before and now, 16 heads of 64 | 4 of 128:
//   861 rows x 3 sequences  232 -> 120 | 287 -> 81        64 x 4   15.2 -> 9.2 | 23 -> 15.6
//   2,580 x 3              1168 -> 820 | 931 -> 440      120 x 4   27 -> 18    | 42 -> 16
//   2,580 x 1               602 -> 296 | 835 -> 205      300 x 2   61 -> 38    | 96 -> 28
template <int HW, int W, int queries, bool Rotary>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2, 4))) void prefill_kernel(
    const uint16_t* __restrict__ qkv, int width, const int* __restrict__ sequence_start,
    const int* __restrict__ sequence_length, const int* __restrict__ sequence_replay,
    const uint16_t* __restrict__ rotations, int heads, int columns, float scale, uint16_t* __restrict__ out)
{
    using Shared = PrefillShared<HW, W, queries>;
    constexpr int per_lane = Shared::per_lane;
    using Weights = float __attribute__((ext_vector_type(per_lane)));
    // With one query a lane, registers hold a block's keys and a half's values, so that
    // their loads wait for memory once.
    constexpr bool ahead = per_lane == 1;
    constexpr int phases = HW / phase_coordinates, held_phases = ahead ? phases : 1;
    constexpr int chunks = tile / chunk_keys, held_chunks = ahead ? chunks : 1;
    constexpr int score_steps = ahead ? 2 : 1, key_steps = ahead ? 8 : 2; // unrolled
    constexpr int q_row = Shared::q_row, k_row = Shared::k_row, p_row = Shared::p_row;
    __shared__ Shared shared;
    const int sequence = blockIdx.x / heads, head = blockIdx.x % heads;
    const int length = sequence_length[sequence];
    // The longest histories first.
    const int q0 = (columns - 1 - int(blockIdx.z * grid_reach + blockIdx.y)) * queries;
    if (q0 < 0 || q0 >= length)
    {
        return;
    }
    const int replay = sequence_replay[sequence];
    const std::size_t stride = std::size_t(3) * width;
    const uint16_t* const base = qkv + std::size_t(sequence_start[sequence]) * stride + head * HW;
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x / 64));
    const int lq = lane / 8, lk = lane % 8;

    for (int i = threadIdx.x; i < queries * HW / 8; i += 64 * W)
    {
        const int r = i / (HW / 8), c = i % (HW / 8), position = q0 + r;
        u32x4 u = u32x4{0, 0, 0, 0};
        if (position < length)
        {
            u = *reinterpret_cast<const u32x4*>(base + std::size_t(position) * stride + c * 8);
            if constexpr (Rotary)
            {
                u = rotate8(u, load16(rotations + std::size_t(position) * HW + c * 8));
            }
        }
        *reinterpret_cast<u32x4*>(shared.q + r * q_row + c * 8) = u;
    }
    // The state before the first block: original_exp(-inf) scales it away.
    for (int i = threadIdx.x; i < HW / 64 * per_lane * 2 * 64; i += 64 * W)
    {
        shared.numerator[i / 64][i % 64] = f32x4{0, 0, 0, 0};
    }
    if (threadIdx.x < queries)
    {
        shared.maximum[threadIdx.x] = -__builtin_inff();
        shared.total[threadIdx.x] = 0.0f;
    }
    if (threadIdx.x < HW / value_coordinates)
    {
        shared.turn[threadIdx.x] = 0;
    }
    __syncthreads();

    typename Shared::Wave& mine = shared.wave[wave];
    const int last_block = (q0 + queries - 1 < length - 1 ? q0 + queries - 1 : length - 1) / tile;
    for (int block = wave; block <= last_block; block += W)
    {
        const int k0 = block * tile;
        // Keys past the sequence read its last one, and are masked out.
        u32x4 held[held_phases][4], held_rotation[held_phases][4] = {};
        const auto fetch_keys = [&](int phase)
        {
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const int i = lane + 64 * j, r = i / 4, c = phase * phase_coordinates + i % 4 * 8;
                const int position = k0 + r < length ? k0 + r : length - 1;
                held[phase % held_phases][j] =
                    *reinterpret_cast<const u32x4*>(base + std::size_t(position) * stride + width + c);
                if constexpr (Rotary)
                {
                    held_rotation[phase % held_phases][j] = load16(rotations + std::size_t(position) * HW + c);
                }
            }
        };
        // Value rows, 16 keys x 64 coordinates at a time: rows past the sequence
        // read its last one, and their weights are never applied.
        u32x4 held_values[held_chunks][2];
        const auto fetch_values = [&](int half, int chunk)
        {
#pragma unroll
            for (int j = 0; j < 2; ++j)
            {
                const int i = lane + 64 * j, r = k0 + chunk * chunk_keys + i / 8;
                const int position = r < length ? r : length - 1;
                held_values[chunk % held_chunks][j] = *reinterpret_cast<const u32x4*>(
                    base + std::size_t(position) * stride + 2 * width + half * value_coordinates + i % 8 * 8);
            }
        };
        const auto fetch_first_values = [&](int half)
        {
#pragma unroll
            for (int chunk = 0; chunk < held_chunks; ++chunk)
            {
                fetch_values(half, chunk);
            }
        };
        float dot[per_lane][8]; // scores, then weights
#pragma unroll
        for (int a = 0; a < per_lane; ++a)
        {
#pragma unroll
            for (int b = 0; b < 8; ++b)
            {
                dot[a][b] = 0.0f;
            }
        }
        const auto score_phase = [&](int phase)
        {
            tile_fence();
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const int i = lane + 64 * j, r = i / 4, c = i % 4;
                *reinterpret_cast<u32x4*>(mine.k + r * k_row + c * 8) =
                    Rotary ? rotate8(held[phase % held_phases][j], held_rotation[phase % held_phases][j])
                           : held[phase % held_phases][j];
            }
            tile_fence();
#pragma unroll score_steps
            for (int c = 0; c < phase_coordinates / 8; ++c)
            {
                u32x4 qu[per_lane], ku[8];
#pragma unroll
                for (int a = 0; a < per_lane; ++a)
                {
                    qu[a] = *reinterpret_cast<const u32x4*>(shared.q + (lq + 8 * a) * q_row +
                                                            phase * phase_coordinates + c * 8);
                }
#pragma unroll
                for (int b = 0; b < 8; ++b)
                {
                    ku[b] = *reinterpret_cast<const u32x4*>(mine.k + (lk + 8 * b) * k_row + c * 8);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e)
                {
                    float qv[per_lane], kv[8];
#pragma unroll
                    for (int a = 0; a < per_lane; ++a)
                    {
                        qv[a] = __uint_as_float(e % 2 ? qu[a][e / 2] & 0xffff0000u : qu[a][e / 2] << 16);
                    }
#pragma unroll
                    for (int b = 0; b < 8; ++b)
                    {
                        kv[b] = __uint_as_float(e % 2 ? ku[b][e / 2] & 0xffff0000u : ku[b][e / 2] << 16);
                    }
#pragma unroll
                    for (int a = 0; a < per_lane; ++a)
                    {
#pragma unroll
                        for (int b = 0; b < 8; ++b)
                        {
                            dot[a][b] = __builtin_fmaf(qv[a], kv[b], dot[a][b]);
                        }
                    }
                }
            }
        };
        if constexpr (ahead)
        {
#pragma unroll
            for (int phase = 0; phase < phases; ++phase)
            {
                fetch_keys(phase);
            }
            fetch_first_values(0);
#pragma unroll
            for (int phase = 0; phase < phases; ++phase)
            {
                score_phase(phase);
            }
        }
        else
        {
            for (int phase = 0; phase < phases; ++phase)
            {
                fetch_keys(phase);
                score_phase(phase);
            }
        }

        if constexpr (!ahead)
        {
            fetch_first_values(0);
        }

        // A query's last live key of the block (all of them but for the last block's).
        int last_key[per_lane];
#pragma unroll
        for (int a = 0; a < per_lane; ++a)
        {
            const int query = q0 + lq + 8 * a;
            last_key[a] = (query < length ? query : length - 1) - k0;
        }
        float block_maximum[per_lane], block_sum[per_lane];
        // Whether every live score lies within 87 of its query's maximum. Then
        // original_exp's clamps and its check change nothing, every weight is 0 or at
        // least exp(-87) > 2^-126, so no sum of them is subnormal and the FTZ tree's
        // flushes change nothing either.
        bool ordinary = true;
#pragma unroll
        for (int a = 0; a < per_lane; ++a)
        {
            float maximum = -__builtin_inff();
#pragma unroll
            for (int b = 0; b < 8; ++b)
            {
                const float score = dot[a][b] * scale;
                dot[a][b] = score;
                const float live = lk + 8 * b <= last_key[a] ? score : -__builtin_inff();
                maximum = maximum < live ? live : maximum;
            }
            maximum = group_max<8>(maximum);
#pragma unroll
            for (int b = 0; b < 8; ++b)
            {
                const float shifted = dot[a][b] - maximum;
                dot[a][b] = shifted;
                ordinary = ordinary & ((lk + 8 * b > last_key[a]) | (shifted >= -87.0f));
            }
            block_maximum[a] = maximum;
        }
        const bool plain = __all(ordinary);
        // Pair tree over the 64 (zero-padded) block positions; for eight or fewer
        // live positions the extra +0 levels leave the eight-wide tree unchanged
        // (src/format/categorical.cpp:44-50).
        const auto weigh = [&](auto exponential, auto tree)
        {
#pragma unroll
            for (int a = 0; a < per_lane; ++a)
            {
                float eighths[8];
#pragma unroll
                for (int b = 0; b < 8; ++b)
                {
                    const float e = exponential(dot[a][b]);
                    dot[a][b] = lk + 8 * b <= last_key[a] ? e : 0.0f;
                    eighths[b] = dot[a][b];
                }
                block_sum[a] = tree(eighths);
                // One query at a time, before the value rows are waited for: all
                // eight at once would spill.
#pragma unroll
                for (int b = 0; b < 8; ++b)
                {
                    asm volatile("" : "+v"(dot[a][b]));
                }
                asm volatile("" : "+v"(block_sum[a]));
            }
        };
        if (plain)
        {
            weigh([](float z) { return exp_within(z); },
                  [](float (&v)[8])
                  {
#pragma unroll
                      for (int b = 0; b < 8; ++b)
                      {
                          v[b] = plain_tree_sum<8>(v[b]);
                      }
                      return register_tree<8, false>(v);
                  });
        }
        else
        {
            weigh([](float z) { return original_exp(z); },
                  [](float (&v)[8])
                  {
#pragma unroll
                      for (int b = 0; b < 8; ++b)
                      {
                          v[b] = tree_sum<8>(v[b]);
                      }
                      return register_tree(v);
                  });
        }

        float old_scale[per_lane], new_scale[per_lane];
#pragma unroll 1
        for (int half = 0; half < HW / value_coordinates; ++half)
        {
            // Value sums: serial fma over each query's live keys, ascending. Dead
            // keys have weight 0, and fma(value, 0, sum) leaves every sum but -0 as it
            // is, unless the value is not finite; the sums of the last block (the only
            // one with dead keys) are made again with those terms left out where one
            // came out zero or NaN.
            float sums[per_lane][8];
            const int last_live = min(q0 + queries - 1, length - 1) - k0; // of any query
            const auto accumulate = [&]<bool Careful>()
            {
#pragma unroll
                for (int a = 0; a < per_lane; ++a)
                {
#pragma unroll
                    for (int c = 0; c < 8; ++c)
                    {
                        sums[a][c] = 0.0f;
                    }
                }
                if (Careful || half > 0)
                {
                    fetch_first_values(half);
                }
#pragma unroll
                for (int chunk = 0; chunk < chunks; ++chunk)
                {
                    if (chunk * chunk_keys > last_live)
                    {
                        break;
                    }
                    tile_fence();
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                    {
                        const int b = chunk * 2 + i;
                        Weights w;
#pragma unroll
                        for (int a = 0; a < per_lane; ++a)
                        {
                            w[a] = dot[a][b];
                        }
                        *reinterpret_cast<Weights*>(mine.p + (lk + 8 * i) * p_row + lq * per_lane) = w;
                        *reinterpret_cast<u32x4*>(mine.v + (lane + 64 * i) * 8) = held_values[chunk % held_chunks][i];
                    }
                    tile_fence();
                    if (!ahead && chunk + 1 < chunks)
                    {
                        fetch_values(half, chunk + 1);
                    }
                    const auto term = [&](int t)
                    {
                        const Weights w = *reinterpret_cast<const Weights*>(mine.p + t * p_row + lq * per_lane);
                        float value[8];
                        widen8(*reinterpret_cast<const u32x4*>(mine.v + t * value_coordinates + lk * 8), value);
#pragma unroll
                        for (int a = 0; a < per_lane; ++a)
                        {
#pragma unroll
                            for (int c = 0; c < 8; ++c)
                            {
                                const float next = __builtin_fmaf(value[c], w[a], sums[a][c]);
                                sums[a][c] = !Careful || chunk * chunk_keys + t <= last_key[a] ? next : sums[a][c];
                            }
                        }
                    };
                    if constexpr (Careful)
                    {
#pragma unroll 1
                        for (int t = 0; t < chunk_keys; ++t)
                        {
                            term(t);
                        }
                    }
                    else
                    {
#pragma unroll key_steps
                        for (int t = 0; t < chunk_keys; ++t)
                        {
                            term(t);
                        }
                    }
                }
            };
            accumulate.template operator()<false>();
            if (block == last_block)
            {
                bool settled = true;
#pragma unroll
                for (int a = 0; a < per_lane; ++a)
                {
#pragma unroll
                    for (int c = 0; c < 8; ++c)
                    {
                        settled = settled & __builtin_islessgreater(sums[a][c], 0.0f);
                    }
                }
                if (!__all(settled))
                {
                    accumulate.template operator()<true>();
                }
            }

            // The running state up to this block.
            while (__hip_atomic_load(&shared.turn[half], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) != block)
            {
                __builtin_amdgcn_s_sleep(1);
            }
            if (half == 0)
            {
#pragma unroll
                for (int a = 0; a < per_lane; ++a)
                {
                    const int q = lq + 8 * a;
                    const float running = shared.maximum[q];
                    const float total = shared.total[q];
                    const float maximum = block_maximum[a];
                    const float factor = original_exp(-__builtin_fabsf(maximum - running));
                    old_scale[a] = running > maximum ? 1.0f : factor;
                    new_scale[a] = running > maximum ? factor : 1.0f;
                    const float old_total = total * old_scale[a];
                    block_sum[a] = __builtin_fmaf(block_sum[a], new_scale[a], old_total);
                    block_maximum[a] = running < maximum ? maximum : running;
                }
                tile_fence(); // every lane has read the row its own lanes now write
#pragma unroll
                for (int a = 0; a < per_lane; ++a)
                {
                    shared.maximum[lq + 8 * a] = block_maximum[a];
                    shared.total[lq + 8 * a] = block_sum[a];
                }
            }
#pragma unroll
            for (int a = 0; a < per_lane; ++a)
            {
                const int query = q0 + lq + 8 * a;
                const bool round_values = query + 1 > 64 || query < replay;
                float numerator[8];
#pragma unroll
                for (int h = 0; h < 2; ++h)
                {
                    const f32x4 n = shared.numerator[(half * per_lane + a) * 2 + h][lane];
                    const float old4[4] = {n.x, n.y, n.z, n.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                    {
                        const int c = h * 4 + i;
                        const float sum = round_values ? round_bf16(sums[a][c]) : sums[a][c];
                        const float old = old4[i] * old_scale[a];
                        numerator[c] = __builtin_fmaf(sum, new_scale[a], old);
                    }
                }
                if (block < last_block)
                {
                    shared.numerator[(half * per_lane + a) * 2][lane] =
                        f32x4{numerator[0], numerator[1], numerator[2], numerator[3]};
                    shared.numerator[(half * per_lane + a) * 2 + 1][lane] =
                        f32x4{numerator[4], numerator[5], numerator[6], numerator[7]};
                }
                else if (query < length)
                {
                    const float reciprocal = 1.0f / block_sum[a];
                    uint32_t words[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                    {
                        words[i] = float_to_bf16(numerator[2 * i] * reciprocal) |
                                   (uint32_t(float_to_bf16(numerator[2 * i + 1] * reciprocal)) << 16);
                    }
                    __builtin_memcpy(out + (std::size_t(sequence_start[sequence]) + query) * width + head * HW +
                                         half * value_coordinates + lk * 8,
                                     words, 16);
                }
            }
            if (lane == 0)
            {
                __hip_atomic_store(&shared.turn[half], block + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }
}

// Sequences of at most 16 rows (the codebook stack's: a frame's books), one wave per
// (sequence, head). Lane (g, t) = (lane / 16, lane % 16) holds the scores of key t
// with queries g + 4 a, so the 16-lane butterfly is the pair tree over the block (its
// higher levels add +0); then lane l holds the value sums of coordinates l (64-wide
// heads) or 2 l and 2 l + 1 of every query. There is one block, merged into the
// empty state by the recurrence all the same.
//
// Bound by HBM: each row of the projection is read once and each output written once.
// 2,580 sequences of 12 rows, 16 heads of 64 (253 MB): 567 us with 64 queries a workgroup,
// 79 here (3.2 TB/s); 4 heads of 128 326 and 36. (On the tiled kernel above, whose waves
// each take a whole 64-key block, 638 and not measured.)
constexpr int short_rows = 16, short_waves = 4;

template <int HW, bool Rotary>
__global__ __launch_bounds__(64 * short_waves) void short_kernel(
    const uint16_t* __restrict__ qkv, int width, const int* __restrict__ sequence_start,
    const int* __restrict__ sequence_length, const int* __restrict__ sequence_replay,
    const uint16_t* __restrict__ rotations, int heads, int pairs, float scale, uint16_t* __restrict__ out)
{
    constexpr int row = HW + 8, chunks = HW / 8, columns = HW / 64;
    constexpr int loads = short_rows * chunks / 64;
    __shared__ __attribute__((aligned(16))) uint16_t tiles[short_waves][2][short_rows * row];
    __shared__ __attribute__((aligned(16))) float weights[short_waves][short_rows][short_rows + 4];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x / 64));
    const int pair = int(blockIdx.x) * short_waves + wave;
    if (pair >= pairs)
    {
        return;
    }
    const int sequence = pair / heads, head = pair % heads;
    const int length = min(sequence_length[sequence], short_rows);
    if (length <= 0)
    {
        return;
    }
    const int replay = sequence_replay[sequence];
    const std::size_t stride = std::size_t(3) * width;
    const std::size_t first = std::size_t(sequence_start[sequence]);
    const uint16_t* const base = qkv + first * stride + head * HW;
    uint16_t* const query_tile = tiles[wave][0];
    uint16_t* const key_tile = tiles[wave][1];

    // Rows past the sequence repeat its last one, and are masked out or not stored.
    u32x4 held[2][loads], held_rotation[loads] = {};
#pragma unroll
    for (int j = 0; j < loads; ++j)
    {
        const int i = lane + 64 * j, r = i / chunks, c = i % chunks * 8;
        const int position = r < length ? r : length - 1;
        const uint16_t* const from = base + std::size_t(position) * stride + c;
        held[0][j] = *reinterpret_cast<const u32x4*>(from);
        held[1][j] = *reinterpret_cast<const u32x4*>(from + width);
        if constexpr (Rotary)
        {
            held_rotation[j] = load16(rotations + std::size_t(position) * HW + c);
        }
    }
    uint32_t values[short_rows]; // the lane's coordinates of each row, BF16
#pragma unroll
    for (int t = 0; t < short_rows; ++t)
    {
        const uint16_t* const from =
            base + std::size_t(t < length ? t : length - 1) * stride + 2 * width + columns * lane;
        if constexpr (columns == 2)
        {
            __builtin_memcpy(&values[t], from, 4);
        }
        else
        {
            values[t] = *from;
        }
    }
#pragma unroll
    for (int j = 0; j < loads; ++j)
    {
        const int i = lane + 64 * j, r = i / chunks, c = i % chunks * 8;
        *reinterpret_cast<u32x4*>(query_tile + r * row + c) =
            Rotary ? rotate8(held[0][j], held_rotation[j]) : held[0][j];
        *reinterpret_cast<u32x4*>(key_tile + r * row + c) =
            Rotary ? rotate8(held[1][j], held_rotation[j]) : held[1][j];
    }
    tile_fence();

    const int g = lane / 16, t = lane % 16;
    float dot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int c = 0; c < chunks; ++c)
    {
        float kv[8], qv[8];
        widen8(*reinterpret_cast<const u32x4*>(key_tile + t * row + c * 8), kv);
#pragma unroll
        for (int a = 0; a < 4; ++a)
        {
            widen8(*reinterpret_cast<const u32x4*>(query_tile + (g + 4 * a) * row + c * 8), qv);
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                dot[a] = __builtin_fmaf(qv[e], kv[e], dot[a]);
            }
        }
    }
    // Each query's weights, and the scales its block joins the empty state with.
    float total[4], old_scale[4], new_scale[4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
    {
        const int query = g + 4 * a;
        const bool live = t <= query && t < length;
        const float score = dot[a] * scale;
        float maximum = -__builtin_inff();
        maximum = live && maximum < score ? score : maximum;
        maximum = group_max<16>(maximum);
        const float e = original_exp(score - maximum);
        const float weight = live ? e : 0.0f;
        weights[wave][query][t] = weight;
        const float sum = tree_sum<16>(weight);
        const float running = -__builtin_inff();
        const float factor = original_exp(-__builtin_fabsf(maximum - running));
        old_scale[a] = running > maximum ? 1.0f : factor;
        new_scale[a] = running > maximum ? factor : 1.0f;
        total[a] = __builtin_fmaf(sum, new_scale[a], 0.0f * old_scale[a]);
    }
    tile_fence();
#pragma unroll
    for (int query = 0; query < short_rows; ++query)
    {
        if (query >= length)
        {
            continue;
        }
        // From a lane of the query's group.
        const int source = query % 4 * 16;
        const float query_total = __shfl(total[query / 4], source), query_old = __shfl(old_scale[query / 4], source),
                    query_new = __shfl(new_scale[query / 4], source);
        float sums[columns];
#pragma unroll
        for (int c = 0; c < columns; ++c)
        {
            sums[c] = 0.0f;
        }
        // Serial fma over the query's live keys, ascending.
#pragma unroll
        for (int key = 0; key < short_rows; ++key)
        {
            if (key > query)
            {
                continue;
            }
            const float weight = weights[wave][query][key];
#pragma unroll
            for (int c = 0; c < columns; ++c)
            {
                const float value = __uint_as_float(c ? values[key] & 0xffff0000u : values[key] << 16);
                sums[c] = __builtin_fmaf(value, weight, sums[c]);
            }
        }
        const float reciprocal = 1.0f / query_total;
        uint32_t word = 0;
#pragma unroll
        for (int c = 0; c < columns; ++c)
        {
            const float sum = query < replay ? round_bf16(sums[c]) : sums[c];
            const float numerator = __builtin_fmaf(sum, query_new, 0.0f * query_old);
            word |= uint32_t(float_to_bf16(numerator * reciprocal)) << (16 * c);
        }
        uint16_t* const to = out + (first + query) * width + head * HW + columns * lane;
        if constexpr (columns == 2)
        {
            __builtin_memcpy(to, &word, 4);
        }
        else
        {
            *to = uint16_t(word);
        }
    }
}
} // namespace

void append_qkv(const uint16_t* qkv, std::size_t rows, std::size_t width, std::size_t head_width,
                const uint16_t* rotation, uint16_t* query, uint16_t* keys, uint16_t* values,
                std::size_t row_stride, hipStream_t stream)
{
    require(width % 2 == 0 && head_width % 2 == 0 && width % head_width == 0, "append: shape");
    if (!rows)
    {
        return;
    }
    const std::size_t n = rows * width / 2;
    const unsigned grid = unsigned((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
    append_kernel<<<grid, 256, 0, stream>>>(qkv, int(rows), int(width), int(head_width), rotation,
                                            query, keys, values, row_stride);
    check_hip(hipGetLastError(), "append launch");
}

namespace
{
__global__ void clear_arrivals(unsigned* words, std::size_t count)
{
    for (std::size_t i = blockIdx.x * std::size_t(blockDim.x) + threadIdx.x; i < count;
         i += std::size_t(gridDim.x) * blockDim.x)
    {
        words[i] = 0;
    }
}
} // namespace

std::size_t decode_partial_floats(std::size_t sequences, std::size_t heads, std::size_t head_width,
                                  std::size_t time)
{
    const std::size_t blocks = (time + 63) / 64;
    // Seven records of padding: the merge reads whole groups of eight.
    return decode_splits(int(blocks)) > 1 ? (sequences * heads * blocks + 7) * (2 + head_width) : 0;
}

std::size_t decode_arrival_counters(std::size_t sequences, std::size_t heads, std::size_t time)
{
    return decode_splits(int((time + 63) / 64)) > 1 ? sequences * heads : 0;
}

void clear_arrival_counters(unsigned* counters, std::size_t count, hipStream_t stream)
{
    if (count)
    {
        const std::size_t groups = (count + 255) / 256;
        clear_arrivals<<<unsigned(groups < 1024 ? groups : 1024), 256, 0, stream>>>(counters, count);
        check_hip(hipGetLastError(), "attention counter clear launch");
    }
}

void attention_decode(const uint16_t* query, const uint16_t* keys, const uint16_t* values,
                      std::size_t sequence_stride, std::size_t sequences, std::size_t time,
                      std::size_t heads, std::size_t head_width, float scale, bool replay,
                      float* partial, unsigned* arrivals, uint16_t* out, hipStream_t stream)
{
    require(time > 0 && sequences > 0, "attention: empty shape");
    require(time < (std::size_t(1) << 30) && sequences * heads < (std::size_t(1) << 24), "attention: shape too large");
    require(head_width == 64 || head_width == 128, "attention: head width must be 64 or 128");
    require(time * heads * head_width * 2 < (std::size_t(1) << 31), "attention: history too long for one decode");
    const int max_blocks = int((time + 63) / 64);
    const int width = int(heads * head_width);
    const int round_values = time > 64 || replay;
    const std::size_t pairs = sequences * heads;
    require(!decode_partial_floats(sequences, heads, head_width, time) || partial != nullptr,
            "attention: this history needs the decode records scratch");
    require(!decode_arrival_counters(sequences, heads, time) || arrivals != nullptr,
            "attention: this history needs the decode arrival counters");
    const int splits = decode_splits(max_blocks);
    require(pairs * splits < (std::size_t(1) << 31), "attention: too many workgroups for one decode");
    // Records stay in LDS only with one split (then with the merge's seven
    // records of padding).
    const std::size_t lds = splits == 1 ? std::size_t(max_blocks + 7) * (2 + head_width) * 4 : 0;
    const unsigned grid = unsigned(pairs * splits);
    const auto launch = [&](auto kernel)
    {
        check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)),
                  "attention decode LDS");
        kernel<<<grid, decode_waves * 64, lds, stream>>>(query, keys, values, sequence_stride, width, int(time),
                                                        int(heads), scale, round_values, partial, arrivals, out);
    };
    if (head_width == 64)
    {
        launch(decode_attention_kernel<64>);
    }
    else
    {
        launch(decode_attention_kernel<128>);
    }
    check_hip(hipGetLastError(), "attention decode launch");
}

void attention_prefill(const uint16_t* qkv, std::size_t width, std::size_t heads,
                       std::size_t head_width, const int* sequence_start,
                       const int* sequence_length, const int* sequence_replay,
                       std::size_t sequences, std::size_t max_length, const uint16_t* rotations,
                       float scale, uint16_t* out, hipStream_t stream)
{
    require(width == heads * head_width, "attention: width mismatch");
    if (!sequences || !max_length)
    {
        return;
    }
    require(head_width == 64 || head_width == 128, "attention: head width must be 64 or 128");
    require(heads > 0 && heads < (std::size_t(1) << 22) && max_length < (std::size_t(1) << 30),
            "attention: heads or rows out of range");
    // A launch takes so many sequences that its work-items along x stay below 2^32.
    const std::size_t slice = (std::size_t(1) << 22) / heads;
    if (max_length <= short_rows)
    {
        const auto kernel = head_width == 64 ? (rotations ? short_kernel<64, true> : short_kernel<64, false>)
                                             : (rotations ? short_kernel<128, true> : short_kernel<128, false>);
        for (std::size_t first = 0; first < sequences; first += slice)
        {
            const std::size_t pairs = std::min(slice, sequences - first) * heads;
            kernel<<<unsigned((pairs + short_waves - 1) / short_waves), 64 * short_waves, 0, stream>>>(
                qkv, int(width), sequence_start + first, sequence_length + first, sequence_replay + first, rotations,
                int(heads), int(pairs), scale, out);
            check_hip(hipGetLastError(), "attention prefill launch");
        }
        return;
    }
    // Waves and queries of a workgroup, by the blocks of the longest history and by how
    // many workgroups there are for the device's units (256). Small query tiles shorten
    // the chain of a block (8 queries: a quarter of the sums a lane, and its loads wait
    // for memory once), which is the time of a launch that leaves units idle; large ones
    // read and rotate a key for more queries; more waves take more blocks at a time, and
    // are idle slots where there are none. us by events around repeated rotated launches,
    // waves x queries, the launched one marked (16 heads of 64, then 4 of 128):
    //   rows x sequences    1x8    4x8    8x8   1x16   2x16   4x32   8x32
    //   64 x 4             9.6*    9.6     15     14     13     19     19
    //   64 x 64             40     53    222    30*     33     41    131
    //   64 x 1000          577    831   3773   380*    401    592   2150
    //   120 x 4             17    18*     31     25     16     21     21
    //   120 x 100          153    293    737   109*    115    203    457
    //   256 x 3             31     31     51     47     29    26*     40
    //   300 x 2             37     29     44     56     34     35    38*
    //   300 x 4             41     49     86     56     35    40*     61
    //   430 x 1             49    27*     37     76     45     39     27
    //   430 x 20           276    402    653    176   184*    257    390
    //   862 x 3            162    194    258    153    114   120*    160
    //   2580 x 1           456    473    552    443    319   298*    338
    //   2580 x 3          1294   1414   1650    834   827*    848    979
    //   64 x 4           15.5*     15     15     24     23     34     33
    //   64 x 64            21*     31     97     26     24     34     60
    //   64 x 1000          270    360   1609   207*    222    349    956
    //   120 x 4             28    16*     16     43     25     35     35
    //   120 x 100           78    133    321     71    64*    109    219
    //   256 x 3             54    21*     30     83     46     39     38
    //   300 x 2             65     29    28*    100     63     61     39
    //   430 x 1             90     30    21*    140     83     67     43
    //   430 x 20           146    183    276    147   107*    129    183
    //   862 x 3            183     93    122    284    147    126    81*
    //   2580 x 1           530    234    259    827    428    328   206*
    //   2580 x 3           692    659    752    841    547   441*    442
    // The lines are drawn through tile counts and do not take every row's best: of 64-wide
    // heads 300 x 2 (1,216 tiles of 8, past the 4 x 8 line at 1,024) would take 29 us on 4 x 8,
    // 120 x 4 and 300 x 4 16 and 35 on 2 x 16.
    //
    // Launches that fill the device many times over run 64-wide heads of up to 5 blocks on
    // workgroups of one wave: no wave holds its slot without a block or waits for its turn.
    // The largest take 32 queries, whose keys are staged and widened once for them; a
    // block costs 1.73 times that of 16 there, so that they pay where the last tiles are
    // nearly full. Longer histories take two waves then: lengths are on the device and
    // the rule sees the longest only, and one long sequence among short ones is a chain of
    // 18 us a block on one wave, 10 on two. us, 64 queries a workgroup (as it was before
    // the blocks went to waves) | 2x16, 1x16, 2x32, 1x32:
    //   128 x 250       276 |   275   256*   297   260      1024 x 200     8763 | 10753 10542  9217*  8793
    //   128 x 1000     1070 |  1184  1131   1195  1052*     2580 x 30      8508 |  9482  8814  8030*  7691
    //   176 x 1000     2043 |  2049  1958*  2277  2005      512 x 400      4746 |  5743  5527  5027*  4697
    //   256 x 250       889 |   909   866    931   833*     65 + 64 x 1000  390 |   428   384*  457    382
    //   256 x 1000     3406 |  3981  3840   3698  3328*     300 + 1 x 500   154 |    77    72   106     91*
    //   320 x 1000     5009 |  6017  5767   5426  4980*     1024 + 12 x 500 375 |   169   222   187*   291
    // Of 128-wide heads only those of up to 96 rows are faster on one wave (65 + 64 x 1000:
    // 221 | 224, 199*; 96 x 1000 572 | 387, 374*; 128 x 1000 636 | 561*, 575).
    const std::size_t units = std::size_t(compute_units());
    constexpr std::integral_constant<int, 1> one;
    constexpr std::integral_constant<int, 2> two;
    constexpr std::integral_constant<int, 4> four;
    constexpr std::integral_constant<int, 8> eight;
    constexpr std::integral_constant<int, 16> sixteen;
    constexpr std::integral_constant<int, 32> thirty_two;
    const std::size_t longest = (max_length + tile - 1) / tile;
    // (query tile, block) pairs of the longest history.
    const auto blocks = [&](std::size_t queries)
    {
        const std::size_t columns = (max_length + queries - 1) / queries, each = tile / queries, full = columns / each;
        return each * full * (full + 1) / 2 + columns % each * (full + 1);
    };
    const std::size_t work = sequences * heads * blocks(32);
    const bool full = 7 * blocks(32) < 4 * blocks(16); // nearly, the last tile of 32 queries
    const auto tiles = [&](std::size_t queries) { return sequences * heads * ((max_length + queries - 1) / queries); };
    const auto launch = [&](auto rotary, auto plain, int waves, std::size_t queries)
    {
        const std::size_t columns = (max_length + queries - 1) / queries;
        for (std::size_t first = 0; first < sequences; first += slice)
        {
            const dim3 grid(unsigned(std::min(slice, sequences - first) * heads),
                            unsigned(std::min<std::size_t>(columns, grid_reach)),
                            unsigned((columns + grid_reach - 1) / grid_reach));
            (rotations ? rotary : plain)<<<grid, 64 * waves, 0, stream>>>(
                qkv, int(width), sequence_start + first, sequence_length + first, sequence_replay + first, rotations,
                int(heads), int(columns), scale, out);
            check_hip(hipGetLastError(), "attention prefill launch");
        }
    };
    const auto by_width = [&](auto head)
    {
        constexpr int HW = decltype(head)::value;
        const auto variant = [&](auto waves, auto queries)
        {
            constexpr int W = decltype(waves)::value, Q = decltype(queries)::value;
            launch(prefill_kernel<HW, W, Q, true>, prefill_kernel<HW, W, Q, false>, W, Q);
        };
        if (max_length <= tile)
        {
            tiles(8) <= 8 * units ? variant(one, eight) : variant(one, sixteen);
        }
        else if (tiles(8) <= 4 * units)
        {
            tiles(8) <= 2 * units && max_length > 4 * tile ? variant(eight, eight) : variant(four, eight);
        }
        else if (longest <= 2 ? tiles(16) >= 9 * units && (HW == 64 || max_length <= 96)
                              : HW == 64 && longest <= 5 && work >= 200 * units)
        {
            if constexpr (HW == 64)
            {
                full && work >= 300 * units ? variant(one, thirty_two) : variant(one, sixteen);
            }
            else
            {
                variant(one, sixteen);
            }
        }
        else if (HW == 64 && longest > 5 && full && work >= 700 * units)
        {
            if constexpr (HW == 64)
            {
                variant(two, thirty_two);
            }
        }
        else if (max_length <= 2 * tile || tiles(16) >= 12 * units ||
                 (tiles(16) >= 8 * units && max_length <= 8 * tile))
        {
            variant(two, sixteen);
        }
        else
        {
            max_length > 4 * tile && tiles(32) < 2 * units ? variant(eight, thirty_two) : variant(four, thirty_two);
        }
    };
    head_width == 64 ? by_width(std::integral_constant<int, 64>{}) : by_width(std::integral_constant<int, 128>{});
}
} // namespace tsac_hip
