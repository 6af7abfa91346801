// The dense elementwise and row-wise steps of the compressed layers, each in
// one pass over memory: the squared ReLU forward and backward, RMSNorm forward
// and backward, and the bias gradients' column sums.
//
// Follows LCT/components/layers.py:16-71,179-222 and LCT/components/ops.py:6-44
// (which leave the fusion to torch.compile).  Every step is bound by memory:
// BF16 in and out, FP32 arithmetic in registers, one rounding where the
// expression in components/layers.py rounds.
#include "pointwise_ops.h"

namespace lct {
namespace {

using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
using u32x2 = __attribute__((ext_vector_type(2))) uint32_t;

__device__ __forceinline__ float low_float(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float high_float(uint32_t pair) {
    return __uint_as_float(pair & 0xFFFF0000u);
}

// ---- squared ReLU
//
// relu(z) and relu(z)^2 from one read of z (ATen: a pass that reads z and
// writes relu, then one that reads it back: 33 us at 8192 x 3072 where this
// takes 23), and in backward grad * 2 relu where relu is not zero, in place,
// with relu^2 for the weight gradient (ATen: 2 * relu, the product, relu == 0,
// the masked fill and the square, 87 us; here 31).  Eight elements per thread
// and access; the grid covers the tensor once.

// relu of both halves; NaN stays NaN, -0 becomes 0.
__device__ __forceinline__ uint32_t relu_pair(uint32_t pair) {
    const float lo = low_float(pair), hi = high_float(pair);
    return (lo <= 0.0f ? 0u : pair & 0xFFFFu) | (hi <= 0.0f ? 0u : pair & 0xFFFF0000u);
}

__device__ __forceinline__ uint32_t square_pair(uint32_t pair) {
    const float lo = low_float(pair), hi = high_float(pair);
    return round_pair_bf16(lo * lo, hi * hi);
}

// bf16(grad * bf16(2 relu)) where relu is not zero, else 0.
__device__ __forceinline__ uint32_t relu_square_grad_pair(uint32_t grad, uint32_t relu) {
    const float lo = low_float(relu), hi = high_float(relu);
    const uint32_t twice = round_pair_bf16(2.0f * lo, 2.0f * hi);
    const uint32_t product = round_pair_bf16(low_float(grad) * low_float(twice),
                                             high_float(grad) * high_float(twice));
    return (lo == 0.0f ? 0u : product & 0xFFFFu) | (hi == 0.0f ? 0u : product & 0xFFFF0000u);
}

__global__ __launch_bounds__(kLanes) void relu_square_kernel(const uint16_t *__restrict__ z,
                                                             uint16_t *__restrict__ relu,
                                                             uint16_t *__restrict__ square,
                                                             int64_t n) {
    const int64_t i = (int64_t{blockIdx.x} * kLanes + threadIdx.x) * 8;
    if (i + 8 <= n) {
        const u32x4 v = *reinterpret_cast<const u32x4 *>(z + i);
        u32x4 r, s;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            r[k] = relu_pair(v[k]);
            s[k] = square_pair(r[k]);
        }
        *reinterpret_cast<u32x4 *>(relu + i) = r;
        *reinterpret_cast<u32x4 *>(square + i) = s;
        return;
    }
    for (int64_t j = i; j < n; ++j) {
        const uint32_t r = relu_pair(z[j]);
        relu[j] = static_cast<uint16_t>(r);
        square[j] = static_cast<uint16_t>(square_pair(r));
    }
}

__global__ __launch_bounds__(kLanes) void relu_square_backward_kernel(
    const uint16_t *__restrict__ relu, uint16_t *__restrict__ grad,
    uint16_t *__restrict__ square, int64_t n) {
    const int64_t i = (int64_t{blockIdx.x} * kLanes + threadIdx.x) * 8;
    if (i + 8 <= n) {
        const u32x4 r = *reinterpret_cast<const u32x4 *>(relu + i);
        const u32x4 g = *reinterpret_cast<const u32x4 *>(grad + i);
        u32x4 d, s;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            d[k] = relu_square_grad_pair(g[k], r[k]);
            s[k] = square_pair(r[k]);
        }
        *reinterpret_cast<u32x4 *>(grad + i) = d;
        *reinterpret_cast<u32x4 *>(square + i) = s;
        return;
    }
    for (int64_t j = i; j < n; ++j) {
        const uint32_t r = relu[j];
        grad[j] = static_cast<uint16_t>(relu_square_grad_pair(grad[j], r));
        square[j] = static_cast<uint16_t>(square_pair(r));
    }
}

// ---- column sums
//
// sums over rows of a BF16 [rows, cols] matrix, in FP32, rounded to BF16.
// Workgroup (x, y) sums rows [y * per, (y + 1) * per) of 64 columns: 8 lanes
// hold a row's 128 bytes, so its 32 rows in flight are whole lines, and about
// 2048 workgroups share the matrix whatever its width (ATen's reduction ran 3
// workgroups for 768 columns and 12 for 3072: 21 and 23 us at 8192 rows; here
// 8.8 and 13.5 with the second launch; per call, host time included, 13 against 20
// to 25).  Where it is called: column_sum_pays in kernels/fused.py.  The partial sums of the row
// groups are added in their order by sum_groups_kernel, so the result does not
// depend on timing.
constexpr int kSumColumns = 64;
constexpr int kSumRows = 32;

__global__ __launch_bounds__(kLanes) void column_sum_kernel(const uint16_t *__restrict__ g,
                                                            int64_t rows, int32_t cols,
                                                            int64_t per,
                                                            float *__restrict__ partials) {
    __shared__ float tile[kSumRows][kSumColumns + 1];
    const int t = threadIdx.x;
    const int part = (t & 7) * 8, slot = t >> 3;
    const int32_t col = static_cast<int32_t>(blockIdx.x) * kSumColumns + part;
    float acc[8] = {};
    if (col < cols) {
        const int64_t first = int64_t{blockIdx.y} * per;
        const int64_t last = first + per < rows ? first + per : rows;
#pragma unroll 4
        for (int64_t r = first + slot; r < last; r += kSumRows) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(g + r * cols + col);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                acc[2 * k] += low_float(v[k]);
                acc[2 * k + 1] += high_float(v[k]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) tile[slot][part + k] = acc[k];
    __syncthreads();
    if (t >= kSumColumns) return;
    const int32_t c = static_cast<int32_t>(blockIdx.x) * kSumColumns + t;
    if (c >= cols) return;
    float sum = 0.0f;
#pragma unroll
    for (int s = 0; s < kSumRows; ++s) sum += tile[s][t];
    partials[int64_t{blockIdx.y} * cols + c] = sum;
}

// out[c] = bf16(sum of partials[g][c] over the groups), as BF16 or as FP32.
constexpr int kGroupThreads = 1024;
constexpr int kGroupWaves = kGroupThreads / kWave;

__global__ __launch_bounds__(kGroupThreads) void sum_groups_kernel(
    const float *__restrict__ partials, int32_t groups, int32_t cols, void *__restrict__ out,
    int32_t out_bf16) {
    __shared__ float tile[kGroupWaves][kSumColumns];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int32_t c = static_cast<int32_t>(blockIdx.x) * kSumColumns + lane;
    float sum = 0.0f;
    if (c < cols) {
#pragma unroll 8
        for (int32_t g = wave; g < groups; g += kGroupWaves) sum += partials[int64_t{g} * cols + c];
    }
    tile[wave][lane] = sum;
    __syncthreads();
    if (wave != 0 || c >= cols) return;
    float total = 0.0f;
#pragma unroll
    for (int w = 0; w < kGroupWaves; ++w) total += tile[w][lane];
    const uint32_t bits = float_to_bf16(total);
    if (out_bf16)
        static_cast<uint16_t *>(out)[c] = static_cast<uint16_t>(bits);
    else
        static_cast<float *>(out)[c] = bf16_to_float(bits);
}

// ---- RMSNorm
//
// One wave per row, whose columns its lanes hold in registers (4 consecutive
// ones per lane and chunk of 256), so a row is read once and its sums are one
// wave reduction: no LDS and no barrier.

__device__ __forceinline__ float wave_sum_float(float v) {
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, kWave);
    return v;
}

template <int kChunks>
struct Row {
    u32x2 v[kChunks];

    __device__ __forceinline__ void load(const uint16_t *row, int32_t cols) {
#pragma unroll
        for (int k = 0; k < kChunks; ++k) {
            const int32_t c = k * 4 * kWave + wave_lane() * 4;
            v[k] = u32x2{0u, 0u};
            if (c < cols) v[k] = *reinterpret_cast<const u32x2 *>(row + c);
        }
    }
};

// Four of the gain's columns, rounded to BF16.
struct Gain4 {
    float v[4];
};

__device__ __forceinline__ Gain4 load_gain(const void *gain, int32_t gain_bf16, int32_t c) {
    Gain4 out;
    if (gain_bf16) {
        const u32x2 q = *reinterpret_cast<const u32x2 *>(static_cast<const uint16_t *>(gain) + c);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            out.v[2 * j] = low_float(q[j]);
            out.v[2 * j + 1] = high_float(q[j]);
        }
    } else {
        const u32x4 q = *reinterpret_cast<const u32x4 *>(static_cast<const float *>(gain) + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) out.v[j] = bf16_to_float(float_to_bf16(__uint_as_float(q[j])));
    }
    return out;
}

constexpr float kEpsilon = 0x1p-23f;          // FP32's, as ATen's when none is given
constexpr int kRowWaves = kLanes / kWave;   // rows in flight per workgroup

// y = bf16(x * rstd * gain), rstd = 1 / sqrt(mean(x^2) + kEpsilon).  A wave has one
// row and reads the gain (from L2) only for its products, so a SIMD holds
// several rows' loads at once: 9 us at 8192 x 768 and 19 at 8192 x 3072
// (ATen's row kernel: 14.5 and 25; waves that keep the gain and walk several
// rows each, one loading ahead: 10.7 and 32 us).
template <int kChunks>
__global__ __launch_bounds__(kLanes) void rms_norm_kernel(const uint16_t *__restrict__ x,
                                                          const void *__restrict__ gain,
                                                          int32_t gain_bf16,
                                                          uint16_t *__restrict__ y,
                                                          float *__restrict__ rstd, int64_t rows,
                                                          int32_t cols) {
    const int64_t r = int64_t{blockIdx.x} * kRowWaves + threadIdx.x / kWave;
    if (r >= rows) return;
    Row<kChunks> row;
    row.load(x + r * cols, cols);
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < kChunks; ++k) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float lo = low_float(row.v[k][j]), hi = high_float(row.v[k][j]);
            sum += lo * lo + hi * hi;
        }
    }
    const float inverse = rsqrtf(wave_sum_float(sum) / static_cast<float>(cols) + kEpsilon);
    if (wave_lane() == 0) rstd[r] = inverse;
#pragma unroll
    for (int k = 0; k < kChunks; ++k) {
        const int32_t c = k * 4 * kWave + wave_lane() * 4;
        if (c >= cols) continue;
        const Gain4 w = load_gain(gain, gain_bf16, c);
        u32x2 out;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            out[j] = round_pair_bf16(low_float(row.v[k][j]) * inverse * w.v[2 * j],
                                     high_float(row.v[k][j]) * inverse * w.v[2 * j + 1]);
        *reinterpret_cast<u32x2 *>(y + r * cols + c) = out;
    }
}

// With h = x * rstd and d = grad * gain: grad_x = bf16(rstd * (d - h * mean(d
// h))), the gain's gradient sum(grad * h) over the rows (FP32 per wave, then
// over the workgroup's waves in LDS, one partial row per workgroup for
// sum_groups_kernel) and, for a following weight gradient, the normalised
// rows bf16(h * gain) of the forward pass.  (ATen: 41 us for the two gradients
// in three launches and 40 us to rebuild the rows in FP32 steps at 8192 x 768;
// here 17.7 in two launches.)  A wave walks rows `waves in the grid` apart with
// the next row's loads in flight, since its sums of the gain's gradient stay in
// registers: 250 of them at 2048 columns, 349 and 460 (accumulation registers
// among them) at 3072 and 4096, one wave per SIMD from 2049 columns on, where
// rows of HBM's bytes still keep it ahead (with the rows rebuilt, us per call
// here | ATen: 27 | 63 at 2048 x 2304, 55 | 230 at 8192 x 3072, 23 | 54 at 1024 x
// 4096, 78 | 302 at 8192 x 4096).
template <int kChunks>
__global__ __launch_bounds__(kLanes) void rms_norm_backward_kernel(
    const uint16_t *__restrict__ grad, const uint16_t *__restrict__ x,
    const float *__restrict__ rstd, const void *__restrict__ gain, int32_t gain_bf16,
    uint16_t *__restrict__ grad_x, uint16_t *__restrict__ normalized,
    float *__restrict__ partials, int64_t rows, int32_t cols) {
    __shared__ float shared[kChunks * 4 * kWave];
    float weight[kChunks][4], acc[kChunks][4];
#pragma unroll
    for (int k = 0; k < kChunks; ++k) {
        const int32_t c = k * 4 * kWave + wave_lane() * 4;
        Gain4 w{};
        if (c < cols) w = load_gain(gain, gain_bf16, c);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            weight[k][j] = w.v[j];
            acc[k][j] = 0.0f;
        }
    }
    const int wave = threadIdx.x / kWave;
    const int64_t stride = int64_t{gridDim.x} * kRowWaves;
    int64_t r = int64_t{blockIdx.x} * kRowWaves + wave;
    Row<kChunks> next_g, next_x;
    float next_rstd = 0.0f;
    if (r < rows) {
        next_g.load(grad + r * cols, cols);
        next_x.load(x + r * cols, cols);
        next_rstd = rstd[r];
    }
    for (; r < rows; r += stride) {
        const Row<kChunks> g = next_g, v = next_x;
        const float inverse = next_rstd;
        if (r + stride < rows) {
            next_g.load(grad + (r + stride) * cols, cols);
            next_x.load(x + (r + stride) * cols, cols);
            next_rstd = rstd[r + stride];
        }
        float dot = 0.0f;
#pragma unroll
        for (int k = 0; k < kChunks; ++k) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t gp = g.v[k][j / 2], xp = v.v[k][j / 2];
                const float gf = (j & 1) ? high_float(gp) : low_float(gp);
                const float h = ((j & 1) ? high_float(xp) : low_float(xp)) * inverse;
                const float gh = gf * h;
                acc[k][j] += gh;
                dot += gh * weight[k][j];
            }
        }
        const float mean = wave_sum_float(dot) / static_cast<float>(cols);
#pragma unroll
        for (int k = 0; k < kChunks; ++k) {
            const int32_t c = k * 4 * kWave + wave_lane() * 4;
            u32x2 dx, out;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float h0 = low_float(v.v[k][j]) * inverse;
                const float h1 = high_float(v.v[k][j]) * inverse;
                const float w0 = weight[k][2 * j], w1 = weight[k][2 * j + 1];
                dx[j] = round_pair_bf16(inverse * (low_float(g.v[k][j]) * w0 - h0 * mean),
                                        inverse * (high_float(g.v[k][j]) * w1 - h1 * mean));
                out[j] = round_pair_bf16(h0 * w0, h1 * w1);
            }
            if (c < cols) {
                *reinterpret_cast<u32x2 *>(grad_x + r * cols + c) = dx;
                if (normalized != nullptr)
                    *reinterpret_cast<u32x2 *>(normalized + r * cols + c) = out;
            }
        }
    }
    // The waves' sums, added in wave order.
    for (int w = 0; w < kRowWaves; ++w) {
        if (w == wave) {
#pragma unroll
            for (int k = 0; k < kChunks; ++k) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float &slot = shared[(k * 4 + j) * kWave + wave_lane()];
                    slot = w == 0 ? acc[k][j] : slot + acc[k][j];
                }
            }
        }
        __syncthreads();
    }
    for (int32_t i = threadIdx.x; i < kChunks * 4 * kWave; i += kLanes) {
        const int32_t lane = i & (kWave - 1), kj = i / kWave;
        const int32_t c = (kj / 4) * 4 * kWave + lane * 4 + (kj & 3);
        if (c < cols) partials[int64_t{blockIdx.x} * cols + c] = shared[i];
    }
}

bool aligned(const void *p, uintptr_t bytes) {
    return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0;
}

constexpr int32_t kMaxColumns = 4096;          // 16 chunks of a row in registers
// A launch has fewer than 2^32 threads.
constexpr int64_t kMaxGroups = (int64_t{1} << 32) / kLanes - 1;
constexpr int64_t kMaxElements = kMaxGroups * kLanes * 8;   // eight per thread
constexpr int64_t kMaxNormRows = kMaxGroups * kRowWaves;    // one per wave
constexpr int64_t kMaxRows = int64_t{1} << 31;              // where the grid does not grow with them

int32_t sum_groups(const float *partials, int32_t groups, int32_t cols, void *out,
                   int32_t out_bf16, hipStream_t stream) {
    sum_groups_kernel<<<(cols + kSumColumns - 1) / kSumColumns, kGroupThreads, 0, stream>>>(
        partials, groups, cols, out, out_bf16);
    return static_cast<int32_t>(hipGetLastError());
}

// Calls launch(integral_constant<chunks>) for the row length.
template <class Launch>
void by_chunks(int32_t cols, Launch launch) {
    const int32_t chunks = (cols + 4 * kWave - 1) / (4 * kWave);
    if (chunks <= 1) launch(std::integral_constant<int, 1>{});
    else if (chunks <= 2) launch(std::integral_constant<int, 2>{});
    else if (chunks <= 3) launch(std::integral_constant<int, 3>{});
    else if (chunks <= 4) launch(std::integral_constant<int, 4>{});
    else if (chunks <= 6) launch(std::integral_constant<int, 6>{});
    else if (chunks <= 8) launch(std::integral_constant<int, 8>{});
    else if (chunks <= 12) launch(std::integral_constant<int, 12>{});
    else launch(std::integral_constant<int, 16>{});
}

}  // namespace
}  // namespace lct

using namespace lct;

extern "C" int32_t lct_relu_square(const void *z, void *relu, void *square, int64_t n,
                                   hipStream_t stream) {
    if (!z || !relu || !square) return LCT_E_NULL;
    if (n <= 0 || n > kMaxElements) return LCT_E_SIZE;
    if (!aligned(z, 16) || !aligned(relu, 16) || !aligned(square, 16)) return LCT_E_ARG;
    const int64_t grid = (n + kLanes * 8 - 1) / (kLanes * 8);
    relu_square_kernel<<<static_cast<uint32_t>(grid), kLanes, 0, stream>>>(
        static_cast<const uint16_t *>(z), static_cast<uint16_t *>(relu),
        static_cast<uint16_t *>(square), n);
    return static_cast<int32_t>(hipGetLastError());
}

extern "C" int32_t lct_relu_square_backward(const void *relu, void *grad, void *square, int64_t n,
                                            hipStream_t stream) {
    if (!relu || !grad || !square) return LCT_E_NULL;
    if (n <= 0 || n > kMaxElements) return LCT_E_SIZE;
    if (!aligned(relu, 16) || !aligned(grad, 16) || !aligned(square, 16)) return LCT_E_ARG;
    const int64_t grid = (n + kLanes * 8 - 1) / (kLanes * 8);
    relu_square_backward_kernel<<<static_cast<uint32_t>(grid), kLanes, 0, stream>>>(
        static_cast<const uint16_t *>(relu), static_cast<uint16_t *>(grad),
        static_cast<uint16_t *>(square), n);
    return static_cast<int32_t>(hipGetLastError());
}

extern "C" int32_t lct_column_sum(const void *g, int64_t rows, int32_t cols, float *partials,
                                  int64_t partial_floats, void *out, int32_t out_bf16,
                                  hipStream_t stream) {
    if (!g || !partials || !out) return LCT_E_NULL;
    if (rows <= 0 || rows > kMaxRows || cols <= 0 || cols > (1 << 20) || partial_floats < cols)
        return LCT_E_SIZE;
    if ((cols & 7) != 0 || !aligned(g, 16)) return LCT_E_ARG;
    const int32_t strips = (cols + kSumColumns - 1) / kSumColumns;
    int64_t groups = 2048 / strips;
    groups = groups < 8 ? 8 : groups > 128 ? 128 : groups;
    const int64_t most = (rows + kSumRows - 1) / kSumRows;
    if (groups > most) groups = most;
    if (groups > partial_floats / cols) groups = partial_floats / cols;
    const int64_t per = (rows + groups - 1) / groups;
    column_sum_kernel<<<dim3(strips, static_cast<uint32_t>(groups)), kLanes, 0, stream>>>(
        static_cast<const uint16_t *>(g), rows, cols, per, partials);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return static_cast<int32_t>(err);
    return sum_groups(partials, static_cast<int32_t>(groups), cols, out, out_bf16, stream);
}

extern "C" int32_t lct_rms_norm(const void *x, const void *gain, int32_t gain_bf16, void *y,
                                float *rstd, int64_t rows, int32_t cols, hipStream_t stream) {
    if (!x || !gain || !y || !rstd) return LCT_E_NULL;
    if (rows <= 0 || rows > kMaxNormRows || cols <= 0 || cols > kMaxColumns) return LCT_E_SIZE;
    if ((cols & 3) != 0 || !aligned(x, 8) || !aligned(y, 8)
        || !aligned(gain, gain_bf16 ? 8 : 16))
        return LCT_E_ARG;
    const uint32_t grid = static_cast<uint32_t>((rows + kRowWaves - 1) / kRowWaves);
    by_chunks(cols, [&](auto chunks) {
        rms_norm_kernel<decltype(chunks)::value><<<grid, kLanes, 0, stream>>>(
            static_cast<const uint16_t *>(x), gain, gain_bf16, static_cast<uint16_t *>(y), rstd,
            rows, cols);
    });
    return static_cast<int32_t>(hipGetLastError());
}

extern "C" int32_t lct_rms_norm_backward(const void *grad, const void *x, const float *rstd,
                                         const void *gain, int32_t gain_bf16, void *grad_x,
                                         void *normalized, float *partials,
                                         int64_t partial_floats, void *grad_gain,
                                         int32_t grad_gain_bf16, int64_t rows, int32_t cols,
                                         hipStream_t stream) {
    if (!grad || !x || !rstd || !gain || !grad_x || !partials || !grad_gain) return LCT_E_NULL;
    if (rows <= 0 || rows > kMaxRows || cols <= 0 || cols > kMaxColumns || partial_floats < cols)
        return LCT_E_SIZE;
    if ((cols & 3) != 0 || !aligned(grad, 8) || !aligned(x, 8) || !aligned(grad_x, 8)
        || !aligned(normalized, 8) || !aligned(gain, gain_bf16 ? 8 : 16))
        return LCT_E_ARG;
    int64_t groups = (rows + kRowWaves - 1) / kRowWaves;
    if (groups > 512) groups = 512;
    if (groups > partial_floats / cols) groups = partial_floats / cols;
    by_chunks(cols, [&](auto chunks) {
        rms_norm_backward_kernel<decltype(chunks)::value>
            <<<static_cast<uint32_t>(groups), kLanes, 0, stream>>>(
                static_cast<const uint16_t *>(grad), static_cast<const uint16_t *>(x), rstd, gain,
                gain_bf16, static_cast<uint16_t *>(grad_x), static_cast<uint16_t *>(normalized),
                partials, rows, cols);
    });
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return static_cast<int32_t>(err);
    return sum_groups(partials, static_cast<int32_t>(groups), cols, grad_gain, grad_gain_bf16,
                      stream);
}
