// Row-wise LayerNorm (one row per workgroup, spread over its waves) and
// softmax (one wavefront per row), BF16 residual adds, GELU and rotary helpers.
#include "kernels.hpp"
#include "row_ops.hpp"

namespace tsac_hip
{
namespace
{
constexpr int rows_per_block = 4;

// One row per workgroup of Waves waves (the row layout of layer_norm_spread,
// which the decode frame step's projections use).
template <int Vw, int Waves>
__global__ __launch_bounds__(Waves * 64) void layer_norm_kernel(const uint16_t* x,
                                                                const uint16_t* __restrict__ gain,
                                                                const uint16_t* __restrict__ bias,
                                                                uint16_t* out)
{
    constexpr int width = Waves * wave * Vw;
    __shared__ float exchange[2 * Waves];
    const int warp = __builtin_amdgcn_readfirstlane(int(threadIdx.x / wave));
    const std::size_t at = std::size_t(blockIdx.x) * width + threadIdx.x * Vw;
    uint16_t v[Vw], g[Vw], b[Vw];
    load_row<Vw>(x + at, v);
    load_row<Vw>(gain + threadIdx.x * Vw, g);
    load_row<Vw>(bias + threadIdx.x * Vw, b);
    layer_norm_spread<Vw, Waves>(v, g, b, warp, exchange);
    store_row<Vw>(out + at, v);
}

// One row per wave, for calls of many rows: no exchange between waves and a row's
// values in 2 V-byte loads (30,960 rows of 1024: 61 us with a row spread over 8 waves, 22).
template <int V>
__global__ __launch_bounds__(256) void layer_norm_wave_kernel(const uint16_t* x, int rows,
                                                              const uint16_t* __restrict__ gain,
                                                              const uint16_t* __restrict__ bias, uint16_t* out)
{
    const int lane = threadIdx.x % wave;
    const int row = blockIdx.x * rows_per_block + threadIdx.x / wave;
    if (row >= rows)
    {
        return;
    }
    const std::size_t at = std::size_t(row) * (wave * V) + lane * V;
    uint16_t v[V];
    load_row<V>(x + at, v);
    layer_norm_lane<V>(v, gain, bias, lane);
    store_row<V>(out + at, v);
}

// src/common/probability.cpp:96-122
template <int V>
__global__ __launch_bounds__(256) void softmax_kernel(const uint16_t* x, int rows, uint16_t* out,
                                                      uint32_t* error)
{
    constexpr int width = wave * V;
    const int lane = threadIdx.x % wave;
    const int row = blockIdx.x * rows_per_block + threadIdx.x / wave;
    if (row >= rows)
    {
        return;
    }
    uint16_t v[V];
    load_row<V>(x + std::size_t(row) * width + lane * V, v);
    float maximum = -__builtin_inff();
    bool finite = true;
#pragma unroll
    for (int i = 0; i < V; ++i)
    {
        const float value = bf16_to_float(v[i]);
        finite = finite && is_finite(value);
        maximum = maximum < value ? value : maximum;
    }
    if (!finite)
    {
        error[0] = error_nonfinite;
    }
    maximum = group_max<wave>(maximum);
    float e[V], leaves[V];
#pragma unroll
    for (int i = 0; i < V; ++i)
    {
        const float shifted = bf16_to_float(v[i]) - maximum;
        e[i] = original_exp(shifted);
        leaves[i] = e[i];
    }
    const float total = row_sum<V>(leaves);
    const float reciprocal = 1.0f / total;
#pragma unroll
    for (int i = 0; i < V; ++i)
    {
        v[i] = float_to_bf16(e[i] * reciprocal);
    }
    store_row<V>(out + std::size_t(row) * width + lane * V, v);
}

// Eight consecutive values of a lane at any 2-byte-aligned address.
constexpr int vector = 8;
__device__ __forceinline__ void load8(const uint16_t* from, uint16_t (&v)[vector])
{
    __builtin_memcpy(v, from, sizeof v);
}
__device__ __forceinline__ void store8(uint16_t* to, const uint16_t (&v)[vector])
{
    __builtin_memcpy(to, v, sizeof v);
}

__global__ void add_kernel(const uint16_t* a, const uint16_t* b, std::size_t count,
                           std::size_t width, std::size_t period, uint16_t* out)
{
    for (std::size_t i = blockIdx.x * std::size_t(blockDim.x) + threadIdx.x; i < count;
         i += std::size_t(gridDim.x) * blockDim.x)
    {
        const std::size_t row = i / width, column = i % width;
        const uint16_t right = b[(row % period) * width + column];
        out[i] = float_to_bf16(bf16_to_float(a[i]) + bf16_to_float(right));
    }
}

// Rows of whole vectors, fewer than 2^31 of them in a call: one vector a thread, in
// 32-bit index arithmetic (30,960 rows of 1024: 68 us value by value with 64-bit
// divisions, 29).
__global__ __launch_bounds__(256) void add_vectors_kernel(const uint16_t* a, const uint16_t* b, unsigned vectors,
                                                         unsigned width, unsigned period, bool wraps, uint16_t* out)
{
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i >= vectors)
    {
        return;
    }
    unsigned from = i;
    if (wraps)
    {
        const unsigned row = i / width;
        from = (row % period) * width + (i - row * width);
    }
    uint16_t left[vector], right[vector];
    load8(a + std::size_t(i) * vector, left);
    load8(b + std::size_t(from) * vector, right);
#pragma unroll
    for (int k = 0; k < vector; ++k)
    {
        left[k] = float_to_bf16(bf16_to_float(left[k]) + bf16_to_float(right[k]));
    }
    store8(out + std::size_t(i) * vector, left);
}

// One vector a thread, the last count % 8 values by the threads after them
// (30,960 x 4096: 222 us value by value, 97).
__global__ __launch_bounds__(256) void gelu_kernel(const uint16_t* x, std::size_t count, uint16_t* out)
{
    const std::size_t vectors = count / vector, end = vectors + count % vector;
    for (std::size_t i = blockIdx.x * std::size_t(256) + threadIdx.x; i < end; i += gridDim.x * std::size_t(256))
    {
        if (i < vectors)
        {
            uint16_t v[vector];
            load8(x + i * vector, v);
#pragma unroll
            for (int k = 0; k < vector; ++k)
            {
                v[k] = gelu_bf16(v[k]);
            }
            store8(out + i * vector, v);
        }
        else
        {
            const std::size_t at = vectors * vector + (i - vectors);
            out[at] = gelu_bf16(x[at]);
        }
    }
}

// src/common/probability.cpp:24-43 over (real, imaginary) pairs.
__global__ void rotary_kernel(const uint16_t* x, const uint16_t* c, std::size_t pairs,
                              uint16_t* out)
{
    for (std::size_t i = blockIdx.x * std::size_t(blockDim.x) + threadIdx.x; i < pairs;
         i += std::size_t(gridDim.x) * blockDim.x)
    {
        const float re = bf16_to_float(x[2 * i]), im = bf16_to_float(x[2 * i + 1]);
        const float cosine = bf16_to_float(c[2 * i]), sine = bf16_to_float(c[2 * i + 1]);
        const float im_sine = im * sine;
        const float re_sine = re * sine;
        out[2 * i] = float_to_bf16(__builtin_fmaf(re, cosine, -im_sine));
        out[2 * i + 1] = float_to_bf16(__builtin_fmaf(im, cosine, re_sine));
    }
}

unsigned grid_for(std::size_t count)
{
    const std::size_t blocks = (count + 255) / 256;
    return unsigned(blocks < 8192 ? (blocks ? blocks : 1) : 8192);
}
} // namespace

void layer_norm_rows(const uint16_t* x, std::size_t rows, std::size_t width, const uint16_t* gain,
                     const uint16_t* bias, uint16_t* out, hipStream_t stream)
{
    if (!rows)
    {
        return;
    }
    require(rows < (std::size_t(1) << 31), "too many rows");
    const dim3 grid(static_cast<unsigned>(rows));
    // A row a wave once that gives every SIMD two (fewer rows end sooner spread
    // over 8 waves).
    if (rows >= 8 * std::size_t(compute_units()))
    {
        const unsigned blocks = unsigned((rows + rows_per_block - 1) / rows_per_block);
        const auto launch = [&](auto kernel) { kernel<<<blocks, 256, 0, stream>>>(x, int(rows), gain, bias, out); };
        switch (width)
        {
        case 256: launch(layer_norm_wave_kernel<4>); break;
        case 512: launch(layer_norm_wave_kernel<8>); break;
        case 1024: launch(layer_norm_wave_kernel<16>); break;
        case 2048: launch(layer_norm_wave_kernel<32>); break;
        default: throw Error("layer norm: width must be one of 256, 512, 1024, 2048");
        }
        check_hip(hipGetLastError(), "layer norm launch");
        return;
    }
    switch (width)
    {
    case 256:
        layer_norm_kernel<1, 4><<<grid, 256, 0, stream>>>(x, gain, bias, out);
        break;
    case 512:
        layer_norm_kernel<1, 8><<<grid, 512, 0, stream>>>(x, gain, bias, out);
        break;
    case 1024:
        layer_norm_kernel<2, 8><<<grid, 512, 0, stream>>>(x, gain, bias, out);
        break;
    case 2048:
        layer_norm_kernel<4, 8><<<grid, 512, 0, stream>>>(x, gain, bias, out);
        break;
    default:
        throw Error("layer norm: width must be one of 256, 512, 1024, 2048");
    }
    check_hip(hipGetLastError(), "layer norm launch");
}

void softmax_rows(const uint16_t* x, std::size_t rows, std::size_t width, uint16_t* out,
                  uint32_t* error, hipStream_t stream)
{
    if (!rows)
    {
        return;
    }
    require(rows < (std::size_t(1) << 31), "too many rows");
    const dim3 grid(unsigned((rows + rows_per_block - 1) / rows_per_block));
    switch (width)
    {
    case 256:
        softmax_kernel<4><<<grid, 256, 0, stream>>>(x, int(rows), out, error);
        break;
    case 512:
        softmax_kernel<8><<<grid, 256, 0, stream>>>(x, int(rows), out, error);
        break;
    case 1024:
        softmax_kernel<16><<<grid, 256, 0, stream>>>(x, int(rows), out, error);
        break;
    case 2048:
        softmax_kernel<32><<<grid, 256, 0, stream>>>(x, int(rows), out, error);
        break;
    default:
        throw Error("softmax: width must be one of 256, 512, 1024, 2048");
    }
    check_hip(hipGetLastError(), "softmax launch");
}

void add_rows(const uint16_t* a, const uint16_t* b, std::size_t rows, std::size_t width,
              std::size_t b_period, uint16_t* out, hipStream_t stream)
{
    require(width > 0 && b_period > 0, "add: empty shape");
    const std::size_t count = rows * width;
    if (!count)
    {
        return;
    }
    if (width % vector == 0 && count / vector < (std::size_t(1) << 31))
    {
        // A period past the rows never wraps, so it need not fit 32 bits.
        const bool wraps = b_period < rows;
        const unsigned vectors = unsigned(count / vector);
        add_vectors_kernel<<<(vectors + 255) / 256, 256, 0, stream>>>(a, b, vectors, unsigned(width / vector),
                                                                      wraps ? unsigned(b_period) : 1u, wraps, out);
    }
    else
    {
        add_kernel<<<grid_for(count), 256, 0, stream>>>(a, b, count, width, b_period, out);
    }
    check_hip(hipGetLastError(), "add launch");
}

void gelu_values(const uint16_t* x, std::size_t count, uint16_t* out, hipStream_t stream)
{
    if (!count)
    {
        return;
    }
    const std::size_t threads = count / vector + count % vector;
    const std::size_t blocks = std::min((threads + 255) / 256, std::size_t(1) << 23); // 2^31 threads
    gelu_kernel<<<unsigned(blocks), 256, 0, stream>>>(x, count, out);
    check_hip(hipGetLastError(), "gelu launch");
}

void rotary_values(const uint16_t* x, const uint16_t* coefficients, std::size_t count,
                   uint16_t* out, hipStream_t stream)
{
    require(count % 2 == 0, "rotary pair shape mismatch");
    if (!count)
    {
        return;
    }
    rotary_kernel<<<grid_for(count / 2), 256, 0, stream>>>(x, coefficients, count / 2, out);
    check_hip(hipGetLastError(), "rotary launch");
}
} // namespace tsac_hip
