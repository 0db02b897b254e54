// DAC convolutions with fused Snake/residual epilogues, and the RVQ encoder
// and decoder (dac.hpp).
#include "dac.hpp"

#include <algorithm>
#include <iterator>

namespace tsac_hip
{
namespace
{
constexpr int lanes = 64;
constexpr int conv_waves = 4;
constexpr int conv_threads = conv_waves * lanes;

// Reads through the constant address space become scalar loads.
template <class T> using constant_ptr = const __attribute__((address_space(4))) T*;

__device__ __forceinline__ float from_bits(uint32_t bits)
{
    return __uint_as_float(bits);
}

// sin(phase)^2 as src/scalar/dsp.cpp:47-84 computes it: quadrant = the
// nearest integer to phase * 2/pi (ties to even), a two-term Cody-Waite
// reduction, then the odd or even minimax polynomial by the quadrant's parity.
// The parity is that of the reference's int32 conversion, which is even for
// every float at or beyond 2^24 (and the indefinite value beyond 2^31).
__device__ __forceinline__ float sine_squared(float phase)
{
    const float reduced = phase * from_bits(0x3f22f983);
    const float quadrant = __builtin_rintf(reduced);
    const bool odd = __builtin_fabsf(quadrant) < 16777216.0f && (int(quadrant) & 1) != 0;
    float x = __builtin_fmaf(quadrant, from_bits(0xbfc90000), phase);
    x = __builtin_fmaf(quadrant, from_bits(0xb9fdaa22), x);
    const float x2 = x * x;
    float value;
    if (!odd)
    {
        float polynomial = __builtin_fmaf(from_bits(0xb94ca1f9), x2, from_bits(0x3c08839e));
        polynomial = __builtin_fmaf(polynomial, x2, from_bits(0xbe2aaaa3));
        const float cube = x * x2;
        value = __builtin_fmaf(cube, polynomial, x);
    }
    else
    {
        float polynomial = __builtin_fmaf(from_bits(0x37ccf5ce), x2, from_bits(0xbab6061a));
        polynomial = __builtin_fmaf(polynomial, x2, from_bits(0x3d2aaaa5));
        polynomial = __builtin_fmaf(polynomial, x2, from_bits(0xbf000000));
        value = __builtin_fmaf(polynomial, x2, 1.0f);
    }
    return value * value;
}

// Snake of src/scalar/dsp.cpp:86-111: y + sin^2(a y) / (a + eps).
__device__ __forceinline__ float snake(float y, float a, bool& finite)
{
    const float phase = a * y;
    finite = finite && __builtin_isfinite(phase);
    const float squared = sine_squared(phase);
    const float denominator = a + from_bits(0x3089705f);
    const float result = y + squared / denominator;
    finite = finite && __builtin_isfinite(result);
    return result;
}

// Rows of a signal through range-checked buffer loads: a lane whose frame is
// outside the signal gets `outside` as its offset and reads 0 (every other offset is
// below 2 GiB, which dac_conv checks). A skipped term and
// an added 0 * w are the same: a sum starts at +0 and no IEEE addition of +0 and a
// zero, or of opposite finite values, gives -0, so adding a zero of either sign
// never changes a sum.
constexpr uint32_t outside = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_buffer(const float* row)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row), 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ float row_load(__amdgpu_buffer_rsrc_t row, uint32_t at)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(row, at, 0, 0));
}

// The launch's arguments, read again where they are used: kept in scalar
// registers over the product loop they would spill.
__device__ __forceinline__ constant_ptr<ConvArgs> arguments()
{
    auto p = (constant_ptr<ConvArgs>)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// Byte offset of frame f in a channel's row from frame `from` on (0 where polyphase).
__device__ __forceinline__ uint32_t frame_offset(const __attribute__((address_space(4))) Strided& s, int f, int from)
{
    const int phases = s.phases;
    const long long at = phases > 1 ? (f % phases) * s.phase + (f / phases) * s.frame : (f - from) * s.frame;
    return uint32_t(at) * 4u;
}

// LDS-only workgroup barrier: the next stage's global loads stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

// N consecutive values a lane reads from a tile row: quads `quad_step` apart
// (or one pair, or one value), so that a wave's lanes read whole lines.
template <int N> __device__ __forceinline__ void read_values(const float* at, int quad_step, float (&v)[N])
{
    if constexpr (N % 4 == 0)
    {
#pragma unroll
        for (int q = 0; q < N / 4; ++q)
        {
            const float4v four = *reinterpret_cast<const float4v*>(at + q * quad_step);
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                v[q * 4 + i] = four[i];
            }
        }
    }
    else if constexpr (N == 2)
    {
        const float2v two = *reinterpret_cast<const float2v*>(at);
        v[0] = two[0];
        v[1] = two[1];
    }
    else
    {
        static_assert(N == 1);
        v[0] = at[0];
    }
}
// Index of value i of a lane among `lanes_across` lanes along one side of a tile.
template <int N> __device__ __forceinline__ int value_index(int lane, int lanes_across, int i)
{
    return N % 4 == 0 ? i / 4 * 4 * lanes_across + lane * 4 + i % 4 : lane * N + i;
}

// A workgroup of 4 waves (WF along the frames): a tile of positions x columns as
// an outer-product over the inputs, lane (lf, lc) of a wave holding FR positions x
// CO columns. A position of an ordinary convolution is an output frame and a
// column an output channel; a transposed one is the same product with kernel /
// stride taps, where position u makes output frames stride * u - padding + r and
// column channel * stride + r, tap j reading frame u - j. KB inputs of one tap at
// a time go through LDS, double-buffered, the next ones' global loads in flight
// over the current products. Every output stays one serial sum, so the tile
// changes no value.
//
// Bound by VALU issue: a product and an addition per term, which no fused or
// matrix instruction may replace. Separate v_mul/v_add reach 70 T
// instructions/s (70 TFLOP/s counting each) on register operands, and only with an
// even number of ready waves per SIMD. Weights as scalar operands with one frame
// per lane stopped at 46-55: each wave waited for its own loads. From LDS both
// operands of 4 x 8 sums cost three 16-byte reads for 64 instructions. Measured,
// before and now: 768 -> 768, kernel 7, 20,672 frames 45.9 -> 50.4 TFLOP/s; 96
// channels, kernel 1, 1.3 M frames 22.8 -> 33.9 (the epilogue's 16-byte stores);
// 1024 -> 1536, kernel 7, 87 frames 468 -> 190 us (stages ahead instead of a wait
// per 16 inputs; one wave a SIMD); 96 -> 2 exit 734 -> 550 us (2 columns instead of
// 16). Counters of the 128 x 64 tile over 2,584 latent frames: 1.7 VALU instructions a
// SIMD and 4 cycles, of the 2 that two waves issue; waits for LDS in 1.6% of the
// waves' time, no bank conflicts.
// sum[j] = sum[j] + x * w[j], the product rounded first. One asm block for up to
// four columns: left to the compiler, a whole input's products are made before
// the first addition, and their registers spill.
template <int N> __device__ __forceinline__ void add_products(float* sum, float x, const float* w)
{
    if constexpr (N == 4)
    {
        float a, b, c, d;
        asm("v_mul_f32 %4, %8, %9\n\tv_mul_f32 %5, %8, %10\n\tv_mul_f32 %6, %8, %11\n\tv_mul_f32 %7, %8, %12\n\t"
            "v_add_f32 %0, %0, %4\n\tv_add_f32 %1, %1, %5\n\tv_add_f32 %2, %2, %6\n\tv_add_f32 %3, %3, %7"
            : "+v"(sum[0]), "+v"(sum[1]), "+v"(sum[2]), "+v"(sum[3]), "=&v"(a), "=&v"(b), "=&v"(c), "=&v"(d)
            : "v"(x), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]));
    }
    else
    {
        float a, b;
        static_assert(N == 2);
        asm("v_mul_f32 %2, %4, %5\n\tv_mul_f32 %3, %4, %6\n\tv_add_f32 %0, %0, %2\n\tv_add_f32 %1, %1, %3"
            : "+v"(sum[0]), "+v"(sum[1]), "=&v"(a), "=&v"(b)
            : "v"(x), "v"(w[0]), "v"(w[1]));
    }
}

template <int FR, int CO, int LF, int WF, int KB> struct Tile
{
    static constexpr int fr = FR, co = CO, lf = LF, wf = WF, kb = KB;
    static constexpr int lc = lanes / LF, wc = conv_waves / WF;
    static constexpr int positions = WF * LF * FR, columns = wc * lc * CO;
};

template <class T, bool Transposed>
__global__ __launch_bounds__(conv_threads) __attribute__((amdgpu_waves_per_eu(4, 4))) void conv_kernel(const ConvArgs)
{
    constexpr int FR = T::fr, CO = T::co, LF = T::lf, LC = T::lc, KB = T::kb, TP = T::positions, TC = T::columns;
    const auto args = arguments();
    const int thread = threadIdx.x, lane = thread % lanes;
    const int wave = __builtin_amdgcn_readfirstlane(thread / lanes);
    const int lf = lane % LF, lc = lane / LF;
    const int columns = args->conv.columns, inputs = args->conv.shape.in;
    const int p0 = int(blockIdx.x) * TP, c0 = int(blockIdx.y) * TC;
    const int taps = Transposed ? args->conv.shape.kernel / args->conv.shape.stride : args->conv.shape.kernel;
    const long long channel = args->x.channel;

    __shared__ __attribute__((aligned(16))) float xs[2][KB][TP];
    __shared__ __attribute__((aligned(16))) float ws[2][KB][TC];

    // Input rows: thread t loads positions t % TP (and every conv_threads-th) of
    // rows t / TP, t / TP + rows, ...
    constexpr int across = TP < conv_threads ? TP : conv_threads, rows = conv_threads / across;
    constexpr int steps = TP / across, passes = (KB + rows - 1) / rows;
    constexpr bool uniform_row = across % lanes == 0;
    const int column = thread % across;
    const int row = uniform_row ? __builtin_amdgcn_readfirstlane(thread / across) : thread / across;
    uint32_t at[steps];
    // The first frame the tile reads, which its offsets count from: the rows of
    // interleaved PCM may span more than an offset holds.
    const auto first_frame = [&](constant_ptr<ConvArgs> now)
    {
        const int least = Transposed ? p0 - (taps - 1) : p0 * now->conv.shape.stride - now->conv.shape.padding;
        return now->x.phases > 1 || least < 0 ? 0 : least;
    };
    const auto offsets = [&](int tap)
    {
        const auto now = arguments();
        const int from = first_frame(now);
        const int step = Transposed ? 1 : now->conv.shape.stride;
        const int origin = Transposed ? -tap : tap * now->conv.shape.dilation - now->conv.shape.padding;
        const int frames = now->frames;
#pragma unroll
        for (int i = 0; i < steps; ++i)
        {
            const int source = (p0 + column + i * across) * step + origin;
            at[i] = source >= 0 && source < frames
                        ? frame_offset(now->x, source, from) + (uniform_row ? 0u : uint32_t(row * int(channel)) * 4u)
                        : outside;
        }
    };
    const float* const first_row = args->x.data + first_frame(args) * args->x.frame + (uniform_row ? row * channel : 0);
    const float* x = first_row;
    float held[passes][steps];
    // Weights: float4s t, t + conv_threads, ... of the stage's KB x TC.
    constexpr int quads = TC >= 4 ? TC / 4 : 1, per = TC >= 4 ? 4 : TC;
    constexpr int weight_loads = (KB * quads + conv_threads - 1) / conv_threads;
    const float* w = args->conv.w + c0;
    float4v held_weights[weight_loads];
    const auto fetch = [&]()
    {
#pragma unroll
        for (int p = 0; p < passes; ++p)
        {
            if (KB % rows == 0 || row + p * rows < KB)
            {
                const __amdgpu_buffer_rsrc_t source = row_buffer(x + p * rows * channel);
#pragma unroll
                for (int i = 0; i < steps; ++i)
                {
                    held[p][i] = row_load(source, at[i]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < weight_loads; ++i)
        {
            const int quad = thread + i * conv_threads;
            const int k = quad / quads, n = quad % quads * per;
            if ((KB * quads % conv_threads == 0 || k < KB) && c0 + n < columns)
            {
                const float* from = w + std::size_t(k) * columns + n;
                if constexpr (per == 4)
                {
                    held_weights[i] = *reinterpret_cast<const float4v*>(from);
                }
                else
                {
#pragma unroll
                    for (int j = 0; j < per; ++j)
                    {
                        held_weights[i][j] = from[j];
                    }
                }
            }
        }
    };
    const auto keep = [&](int buffer)
    {
#pragma unroll
        for (int p = 0; p < passes; ++p)
        {
            if (KB % rows == 0 || row + p * rows < KB)
            {
#pragma unroll
                for (int i = 0; i < steps; ++i)
                {
                    xs[buffer][p * rows + row][column + i * across] = held[p][i];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < weight_loads; ++i)
        {
            const int quad = thread + i * conv_threads;
            const int k = quad / quads, n = quad % quads * per;
            if (KB * quads % conv_threads == 0 || k < KB)
            {
                if constexpr (per == 4)
                {
                    *reinterpret_cast<float4v*>(&ws[buffer][k][n]) = held_weights[i];
                }
                else
                {
#pragma unroll
                    for (int j = 0; j < per; ++j)
                    {
                        ws[buffer][k][n + j] = held_weights[i][j];
                    }
                }
            }
        }
    };

    float sum[FR][CO];
#pragma unroll
    for (int i = 0; i < FR; ++i)
    {
#pragma unroll
        for (int j = 0; j < CO; ++j)
        {
            sum[i][j] = 0.0f;
        }
    }
    const int wave_position = wave % T::wf * (LF * FR), wave_column = wave / T::wf * (LC * CO);
    const int x_at = wave_position + value_index<FR>(lf, LF, 0), w_at = wave_column + value_index<CO>(lc, LC, 0);
    const int stages = taps * (inputs / KB);
    int tap = 0, input = 0;
    offsets(0);
    fetch();
    keep(0);
    lds_barrier();
    for (int stage = 0; stage < stages; ++stage)
    {
        const int buffer = stage & 1;
        const bool more = stage + 1 < stages;
        if (more)
        {
            input += KB;
            x += KB * channel;
            w += std::size_t(KB) * columns;
            if (input == inputs)
            {
                input = 0;
                x = first_row;
                offsets(++tap);
            }
            fetch();
        }
        // An input's values are read while the previous one's products are made;
        // the fences keep the compiler from reading the whole stage ahead, which
        // would spill.
        float xv[2][FR], wv[2][CO];
        const auto read = [&](int k)
        {
            read_values<FR>(&xs[buffer][k][x_at], 4 * LF, xv[k % 2]);
            read_values<CO>(&ws[buffer][k][w_at], 4 * LC, wv[k % 2]);
        };
        read(0);
#pragma unroll
        for (int k = 0; k < KB; ++k)
        {
            if (k + 1 < KB)
            {
                read(k + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < FR; ++i)
            {
#pragma unroll
                for (int j = 0; j < CO; j += CO % 4 ? 2 : 4)
                {
                    add_products<CO % 4 ? 2 : 4>(&sum[i][j], xv[k % 2][i], &wv[k % 2][j]);
                }
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more)
        {
            keep(buffer ^ 1);
            lds_barrier();
        }
    }

    const auto end = arguments();
    const ConvShape s = {end->conv.shape.in,      end->conv.shape.out,      end->conv.shape.kernel,
                         end->conv.shape.stride,  end->conv.shape.padding,  end->conv.shape.dilation,
                         end->conv.shape.transposed};
    const int out_frames = s.output_frames(end->frames);
    const int low = end->first > 0 ? end->first : 0, high = end->last < out_frames ? end->last : out_frames;
    const int stride = Transposed ? s.stride : 1;
    const int origin = Transposed ? -s.padding : 0;
    float* const out = end->out.data;
    float* const activated = end->activated.data;
    const float* const residual = end->residual.data;
    const float* const bias = end->conv.bias;
    const float* const alpha = end->alpha;
    const long long out_channel = end->out.channel, out_frame = end->out.frame;
    const long long activated_channel = end->activated.channel, activated_frame = end->activated.frame;
    // Polyphase planes are a power of two in number (dac_conv checks it).
    const int phase_mask = end->activated.phases - 1, phase_shift = __builtin_popcount(phase_mask);
    const long long phase = end->activated.phase;
    const bool out_unit = out_frame == 1, activated_unit = activated_frame == 1 && phase_mask == 0;
    bool finite = true;
    // N outputs of channel c from frame f on.
    const auto emit = [&]<int N>(int c, int f, const float (&v)[N])
    {
        if (c >= s.out)
        {
            return;
        }
        const bool whole = N == 4 && f >= low && f + N <= high;
        const float b = bias[c];
        const long long out_at = c * out_channel + f * out_frame;
        float y[N];
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
            y[i] = v[i] + b;
        }
        if (residual)
        {
            if (whole && out_unit)
            {
                const float4u four = *reinterpret_cast<const float4u*>(residual + out_at);
#pragma unroll
                for (int i = 0; i < N; ++i)
                {
                    y[i] = four[i] + y[i];
                }
            }
            else
            {
#pragma unroll
                for (int i = 0; i < N; ++i)
                {
                    if (f + i >= low && f + i < high)
                    {
                        y[i] = residual[out_at + i * out_frame] + y[i];
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
            finite = finite && (__builtin_isfinite(y[i]) || f + i < low || f + i >= high);
        }
        if (out)
        {
            if (whole && out_unit)
            {
                float4u four;
#pragma unroll
                for (int i = 0; i < N; ++i)
                {
                    four[i] = y[i];
                }
                *reinterpret_cast<float4u*>(out + out_at) = four;
            }
            else
            {
#pragma unroll
                for (int i = 0; i < N; ++i)
                {
                    if (f + i >= low && f + i < high)
                    {
                        out[out_at + i * out_frame] = y[i];
                    }
                }
            }
        }
        if (activated)
        {
            const float a = alpha[c];
            float* const to = activated + c * activated_channel;
            float z[N];
#pragma unroll
            for (int i = 0; i < N; ++i)
            {
                bool fits = true;
                z[i] = snake(y[i], a, fits);
                finite = finite && (fits || f + i < low || f + i >= high);
            }
            if (whole && activated_unit)
            {
                float4u four;
#pragma unroll
                for (int i = 0; i < N; ++i)
                {
                    four[i] = z[i];
                }
                *reinterpret_cast<float4u*>(to + f) = four;
            }
            else
            {
#pragma unroll
                for (int i = 0; i < N; ++i)
                {
                    if (f + i >= low && f + i < high)
                    {
                        to[((f + i) & phase_mask) * phase + ((f + i) >> phase_shift) * activated_frame] = z[i];
                    }
                }
            }
        }
        asm volatile("" ::: "memory"); // one run at a time: several at once would spill
    };
    const int u0 = p0 + wave_position, n0 = c0 + wave_column;
    if constexpr (FR % 4 == 0 && CO % 4 == 0)
    {
        // 4 positions x 4 columns a time, as runs of four consecutive output frames.
#pragma unroll
        for (int j = 0; j < CO; j += 4)
        {
#pragma unroll
            for (int i = 0; i < FR; i += 4)
            {
                const int u = u0 + value_index<FR>(lf, LF, i), n = n0 + value_index<CO>(lc, LC, j);
                if constexpr (!Transposed)
                {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                    {
                        emit(n + q, u, {sum[i][j + q], sum[i + 1][j + q], sum[i + 2][j + q], sum[i + 3][j + q]});
                    }
                }
                else if (stride % 4 == 0)
                {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                    {
                        emit(n / stride, (u + q) * stride + origin + n % stride,
                             {sum[i + q][j], sum[i + q][j + 1], sum[i + q][j + 2], sum[i + q][j + 3]});
                    }
                }
                else
                {
                    // stride 2: two channels, each two runs
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                    {
                        const int p = i + q / 2 * 2, k = j + q % 2 * 2;
                        emit(n / 2 + q % 2, (u + q / 2 * 2) * 2 + origin,
                             {sum[p][k], sum[p][k + 1], sum[p + 1][k], sum[p + 1][k + 1]});
                    }
                }
            }
        }
    }
    else
    {
#pragma unroll
        for (int j = 0; j < CO; ++j)
        {
            const int n = n0 + value_index<CO>(lc, LC, j);
            const int c = n / stride, r = n % stride;
#pragma unroll
            for (int i = 0; i < FR; ++i)
            {
                emit(c, (u0 + value_index<FR>(lf, LF, i)) * stride + origin + r, {sum[i][j]});
            }
        }
    }
    if (!finite)
    {
        end->error[0] = 1u;
    }
}

// ---------------------------------------------------------------- RVQ

__device__ __forceinline__ float shuffle(float v, int source)
{
    return __shfl(v, source, lanes);
}

// One wave per frame: the codebooks in order, each its input projection (an
// ordinary 1024 -> 8 pointwise convolution: serial sums over the inputs, then
// the bias), the normalised search (src/weights/preparation.cpp:62-84 and
// src/common/rvq.cpp:131-151) and the chosen vector's projection subtracted
// from the residual (src/common/rvq.tpp:40-57).
__global__ __launch_bounds__(lanes) void rvq_encode_kernel(const RvqBook* books, int count, const float* latent,
                                                         long long stride, int frames, uint16_t* tokens,
                                                         int token_stride, uint32_t* error)
{
    __shared__ float residual[1024];
    const int frame = blockIdx.x, lane = threadIdx.x;
    if (frame >= frames)
    {
        return;
    }
    bool finite = true;
    for (int i = lane; i < 1024; i += lanes)
    {
        residual[i] = latent[i * stride + frame];
        finite = finite && __builtin_isfinite(residual[i]);
    }
    __syncthreads();
    for (int b = 0; b < count; ++b)
    {
        const RvqBook book = books[b];
        float projected = 0.0f;
        if (lane < 8)
        {
            const float* w = book.input_weights + lane * 1024;
            for (int i = 0; i < 1024; ++i)
            {
                const float product = residual[i] * w[i];
                projected = projected + product;
            }
            projected = projected + book.input_bias[lane];
        }
        float q[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
        {
            q[i] = shuffle(projected, i);
            finite = finite && __builtin_isfinite(q[i]);
        }
        // normalize_search: squares reduced by adjacent pairs, RMS with epsilon, 1/sqrt(8).
        float squares[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
        {
            squares[i] = q[i] * q[i];
        }
#pragma unroll
        for (int width = 8; width > 1; width /= 2)
        {
#pragma unroll
            for (int i = 0; i < width / 2; ++i)
            {
                squares[i] = squares[2 * i] + squares[2 * i + 1];
            }
        }
        const float mean = squares[0] * (1.0f / 8.0f);
        const float inverse_rms = 1.0f / __builtin_sqrtf(mean + from_bits(0x2b8cbccc));
        const float inverse_width = 1.0f / __builtin_sqrtf(8.0f);
        float query[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
        {
            const float normalized = q[i] * inverse_rms;
            query[i] = normalized * inverse_width;
        }
        // Each lane scans its entries in ascending order with a strict >, so it
        // keeps its first maximum; the lanes' winners then merge to the largest
        // value, the lowest index among equals: the serial scan's choice.
        float best = -__builtin_inff();
        int chosen = 1024;
        for (int e = lane; e < 1024; e += lanes)
        {
            float similarity = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i)
            {
                similarity = __builtin_fmaf(book.search[e * 8 + i], query[i], similarity);
            }
            if (similarity > best)
            {
                best = similarity;
                chosen = e;
            }
        }
#pragma unroll
        for (int offset = 1; offset < lanes; offset *= 2)
        {
            const float other = __shfl_xor(best, offset, lanes);
            const int other_index = __shfl_xor(chosen, offset, lanes);
            if (other > best || (other == best && other_index < chosen))
            {
                best = other;
                chosen = other_index;
            }
        }
        const int token = chosen >= 1024 ? 0 : chosen;
        if (lane == 0)
        {
            tokens[std::size_t(frame) * token_stride + b] = uint16_t(token);
        }
        __syncthreads(); // every lane has read the residual for the projection above
        float vector[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
        {
            vector[i] = book.codebook[token * 8 + i];
        }
        for (int j = lane; j < 1024; j += lanes)
        {
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i)
            {
                sum = __builtin_fmaf(book.output_weights[j * 8 + i], vector[i], sum);
            }
            residual[j] = residual[j] - (sum + book.output_bias[j]);
            finite = finite && __builtin_isfinite(residual[j]);
        }
        __syncthreads();
    }
    if (!finite)
    {
        error[0] = 1u;
    }
}

// latent[j][frame] = 0 + the books' projections in book order (src/common/rvq.cpp:84-127).
__global__ __launch_bounds__(256) void rvq_decode_kernel(const RvqBook* books, int count, const uint16_t* tokens,
                                                        int token_stride, int frames, float* latent,
                                                        long long stride, uint32_t* error)
{
    const int j = blockIdx.y * 256 + threadIdx.x, frame = blockIdx.x;
    if (j >= 1024 || frame >= frames)
    {
        return;
    }
    float value = 0.0f;
    for (int b = 0; b < count; ++b)
    {
        const RvqBook book = books[b];
        const int token = tokens[std::size_t(frame) * token_stride + b];
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i)
        {
            sum = __builtin_fmaf(book.output_weights[j * 8 + i], book.codebook[token * 8 + i], sum);
        }
        value = value + (sum + book.output_bias[j]);
    }
    latent[j * stride + frame] = value;
    if (!__builtin_isfinite(value))
    {
        error[0] = 1u;
    }
}
} // namespace

void dac_conv_layout(const ConvShape& s, const float* stored, float* out, int columns)
{
    // A transposed convolution's tap j * stride + r of channel o is column
    // o * stride + r of tap j.
    const int stride = s.transposed ? s.stride : 1, taps = s.kernel / stride;
    std::fill(out, out + std::size_t(taps) * s.in * columns, 0.0f);
    for (int tap = 0; tap < s.kernel; ++tap)
    {
        for (int i = 0; i < s.in; ++i)
        {
            for (int o = 0; o < s.out; ++o)
            {
                const std::size_t index = s.transposed ? o + std::size_t(tap) * s.out + std::size_t(i) * s.out * s.kernel
                                                       : i + std::size_t(tap) * s.in + std::size_t(o) * s.in * s.kernel;
                out[(std::size_t(tap / stride) * s.in + i) * columns + o * stride + tap % stride] = stored[index];
            }
        }
    }
}

void dac_conv(const ConvArgs& a, hipStream_t stream)
{
    const ConvShape& s = a.conv.shape;
    require(a.frames > 0 && a.x.data && a.error && (a.out.data || a.activated.data), "dac convolution: arguments");
    require(!a.activated.data || a.alpha, "dac convolution: Snake needs its alpha");
    require(a.conv.columns == dac_conv_columns(s), "dac convolution: layout");
    require(!s.transposed || (s.dilation == 1 && s.kernel % s.stride == 0),
            "dac convolution: a transposed convolution's kernel is a multiple of its stride");
    require(a.x.phases >= 1 && a.activated.phases >= 1 && a.out.phases == 1 && a.residual.phases == 1,
            "dac convolution: only the input and the Snake output may be polyphase");
    require(a.x.phases == 1 || a.frames % a.x.phases == 0, "dac convolution: whole polyphase planes");
    require((a.activated.phases & (a.activated.phases - 1)) == 0, "dac convolution: a power of two of planes");
    require(!s.transposed || s.stride == 2 || s.stride % 4 == 0, "dac convolution: transposed stride");
    require(!a.residual.data || (a.residual.channel == a.out.channel && a.residual.frame == a.out.frame),
            "dac convolution: the residual is laid out as the output");
    // What a tile of at most `widest` positions reads of a channel, or of polyphase
    // planes the whole channel.
    constexpr int widest = 256;
    const long long reads = s.transposed ? widest + s.kernel / s.stride - 1
                                         : (widest - 1) * s.stride + (s.kernel - 1) * s.dilation + 1;
    const long long extent = a.x.phases > 1
                                 ? (a.x.phases - 1) * a.x.phase + (a.frames / a.x.phases - 1) * a.x.frame
                                 : (std::min<long long>(reads, a.frames) - 1) * a.x.frame;
    require(extent >= 0 && extent < (1ll << 29) - 1, "dac convolution: a tile's frames span 2 GiB");
    const int out_frames = s.output_frames(a.frames);
    require(out_frames > 0, "dac convolution has no output frames");
    const int positions = s.transposed ? (out_frames + s.padding + s.stride - 1) / s.stride : out_frames;
    const int columns = s.transposed ? s.out * s.stride : s.out; // without the weights' padding
    const auto launch = [&](auto tile)
    {
        using T = decltype(tile);
        static_assert(T::positions <= widest);
        require(s.in % T::kb == 0, "dac convolution: inputs are a multiple of the stage");
        const dim3 grid(unsigned((positions + T::positions - 1) / T::positions),
                        unsigned((columns + T::columns - 1) / T::columns));
        const auto kernel = s.transposed ? conv_kernel<T, true> : conv_kernel<T, false>;
        kernel<<<grid, conv_threads, 0, stream>>>(a);
    };
    if (s.in % 32)
    {
        // The entry convolution of one or two PCM channels.
        s.in % 2 ? launch(Tile<4, 8, 16, 2, 1>{}) : launch(Tile<4, 8, 16, 2, 2>{});
    }
    else if (columns <= 2)
    {
        // The exit convolution: a tile as wide as its one or two channels.
        launch(Tile<1, 2, 64, 4, 16>{});
    }
    else
    {
        // The tile that should end first: its outputs over the rate it reaches
        // where the grid fills the device (relative, measured on the codec's layers:
        // 128 x 64 56 TFLOP/s, 32 x 16 25), times the rounds of workgroups. A SIMD
        // issues at half rate from one wave, so up to two workgroups of a compute
        // unit take the time of one.
        const std::size_t units = compute_units();
        const auto cost = [&](int tile_positions, int tile_columns, double rate)
        {
            const std::size_t groups = std::size_t((positions + tile_positions - 1) / tile_positions) *
                                       std::size_t((columns + tile_columns - 1) / tile_columns);
            const std::size_t rounds = std::max<std::size_t>(2, (groups + units - 1) / units);
            return double(rounds) * tile_positions * tile_columns / rate;
        };
        // Tiles under 64 positions add a row to the lanes' offsets.
        const bool narrow = a.x.channel < (1ll << 24) && extent < (1ll << 28);
        const double costs[] = {cost(128, 64, 1.0),  cost(256, 32, 0.97), cost(64, 64, 0.96), cost(128, 32, 0.94),
                                cost(64, 32, 0.82), narrow ? cost(32, 32, 0.65) : 1e30,
                                narrow ? cost(32, 16, 0.45) : 1e30};
        switch (std::min_element(std::begin(costs), std::end(costs)) - std::begin(costs))
        {
        case 0: launch(Tile<4, 8, 16, 2, 16>{}); break;
        case 1: launch(Tile<4, 8, 16, 4, 16>{}); break;
        case 2: launch(Tile<4, 4, 16, 1, 32>{}); break;
        case 3: launch(Tile<4, 4, 16, 2, 16>{}); break;
        case 4: launch(Tile<4, 2, 16, 1, 32>{}); break;
        case 5: launch(Tile<2, 2, 16, 1, 32>{}); break;
        default: launch(Tile<1, 2, 32, 1, 32>{}); break;
        }
    }
    check_hip(hipGetLastError(), "dac convolution launch");
}

void rvq_encode(const RvqBook* books, int count, const float* latent, long long stride, int frames, uint16_t* tokens,
                int token_stride, uint32_t* error, hipStream_t stream)
{
    require(count >= 1 && count <= 12 && frames >= 0, "rvq encode: arguments");
    if (!frames)
    {
        return;
    }
    rvq_encode_kernel<<<unsigned(frames), lanes, 0, stream>>>(books, count, latent, stride, frames, tokens,
                                                             token_stride, error);
    check_hip(hipGetLastError(), "rvq encode launch");
}

void rvq_decode(const RvqBook* books, int count, const uint16_t* tokens, int token_stride, int frames, float* latent,
                long long stride, uint32_t* error, hipStream_t stream)
{
    require(count >= 1 && count <= 12 && frames >= 0, "rvq decode: arguments");
    if (!frames)
    {
        return;
    }
    rvq_decode_kernel<<<dim3(unsigned(frames), 4), 256, 0, stream>>>(books, count, tokens, token_stride, frames,
                                                                    latent, stride, error);
    check_hip(hipGetLastError(), "rvq decode launch");
}
} // namespace tsac_hip
