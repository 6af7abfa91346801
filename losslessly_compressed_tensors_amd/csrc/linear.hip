// A @ W^T for up to 16 rows of A and a dense BF16 W: the product behind a
// decode step's tokens.
//
// Follows LCT/operations.py:31-48 (A_compBT), which leaves the product to the
// device's library.  W is read once and the work is nothing beside that read,
// so the kernel is a stream of W with the matrix cores behind it: a workgroup
// takes kTiles x 16 of W's rows, its 8 waves an eighth of the columns each,
// every lane loading 16 bytes of a row straight into an operand register
// (16x16x32 tiles; no LDS on the way), four steps of the columns at a time.
// The waves' FP32 sums meet in LDS and are rounded once.  At 16 rows and W in
// HBM: 23.4 us for 11008 x 4096, 27.6 for 4096 x 11008 and 10.2 for 4096 x 4096
// (the library's product: 25.1, 36.7 and 12.0), of which the read of W at the
// 6.9 TB/s that a plain read reaches is 13, 13 and 5.  Loading the next four
// steps during the product made no difference.  From 17 rows on the library's
// tiles, which share A's loads, are faster.  Fewer rows and smaller weights, us
// per call here | library, W rotating over four to six: 9.7 | 21 from 64 x 64 to
// 8192 x 2048 at 1 to 16 rows (host time), 15.7 | 21 at one row of 32768 x 1024,
// 21.5 | 26.4 at one of 11008 x 4096, 19.6 | 38.5 at one of 4096 x 11008, 53.7 |
// 63.8 at one and 60.0 | 68.8 at 16 of 16384 x 8192.
#include "lct_device.h"

namespace lct {
namespace {

using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using f32x4 = __attribute__((ext_vector_type(4))) float;
using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;

constexpr int kSplit = 8;                    // waves per workgroup, shares of the columns
constexpr int kTile = 16;                    // rows of A, rows of W per tile
constexpr int kStep = 32;                    // columns per matrix instruction
constexpr int kAhead = 4;                    // steps in flight
constexpr int kLinearThreads = kSplit * kWave;

// One group of kAhead steps' operands.
template <int kTiles>
struct Operands {
    u32x4 a[kAhead], w[kAhead][kTiles];

    // Steps [s, s + kAhead) below `end`; zeros past it and past the columns
    // (a multiple of 8).
    __device__ __forceinline__ void load(const uint16_t *a_row, const uint16_t *const (&w_row)[kTiles],
                                         int32_t s, int32_t end, int32_t cols) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            const int32_t c = (s + k) * kStep + (wave_lane() >> 4) * 8;
            const bool here = s + k < end && c < cols;
#pragma unroll
            for (int n = 0; n < kTiles; ++n) {
                w[k][n] = u32x4{0u, 0u, 0u, 0u};
                if (here) w[k][n] = *reinterpret_cast<const u32x4 *>(w_row[n] + c);
            }
            a[k] = u32x4{0u, 0u, 0u, 0u};
            if (here) a[k] = *reinterpret_cast<const u32x4 *>(a_row + c);
        }
    }

    __device__ __forceinline__ void multiply(f32x4 (&acc)[kTiles]) const {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
#pragma unroll
            for (int n = 0; n < kTiles; ++n)
                acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, a[k]), __builtin_bit_cast(bf16x8, w[k][n]), acc[n],
                    0, 0, 0);
        }
    }
};

template <int kTiles>
__global__ __launch_bounds__(kLinearThreads) void skinny_linear_kernel(
    const uint16_t *__restrict__ a, const uint16_t *__restrict__ w, uint16_t *__restrict__ out,
    int32_t tokens, int32_t rows, int32_t cols) {
    __shared__ f32x4 sums[kSplit][kTiles][kWave];
    const int lane = wave_lane(), wave = threadIdx.x / kWave;
    const int32_t first_row = static_cast<int32_t>(blockIdx.x) * (kTiles * kTile);
    // Rows past the end read the last one; their results are not stored.
    const uint16_t *a_row = a + int64_t{min(lane & 15, tokens - 1)} * cols;
    const uint16_t *w_row[kTiles];
    f32x4 acc[kTiles];
#pragma unroll
    for (int n = 0; n < kTiles; ++n) {
        w_row[n] = w + int64_t{min(first_row + n * kTile + (lane & 15), rows - 1)} * cols;
        acc[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const int32_t steps = (cols + kStep - 1) / kStep;
    const int32_t per = (steps + kSplit - 1) / kSplit;
    const int32_t end = min(steps, (wave + 1) * per);
    for (int32_t s = wave * per; s < end; s += kAhead) {
        Operands<kTiles> group;
        group.load(a_row, w_row, s, end, cols);
        group.multiply(acc);
    }
#pragma unroll
    for (int n = 0; n < kTiles; ++n) sums[wave][n][lane] = acc[n];
    __syncthreads();
    // Lane l of a tile's sums holds column l % 16 (W's row) of A's rows
    // 4 (l / 16) .. + 3.
    for (int i = threadIdx.x; i < kTiles * kTile * kTile; i += kLinearThreads) {
        const int n = i % (kTiles * kTile), token = i / (kTiles * kTile);
        const int source = (n & 15) + 16 * (token >> 2);
        float sum = 0.0f;
#pragma unroll
        for (int k = 0; k < kSplit; ++k) sum += sums[k][n / kTile][source][token & 3];
        const int32_t row = first_row + n;
        if (token < tokens && row < rows)
            out[int64_t{token} * rows + row] = static_cast<uint16_t>(float_to_bf16(sum));
    }
}

template <int kTiles>
int32_t launch_skinny(const void *a, const void *w, void *out, int32_t tokens, int32_t rows,
                      int32_t cols, hipStream_t stream) {
    const uint32_t grid = static_cast<uint32_t>((rows + kTiles * kTile - 1) / (kTiles * kTile));
    skinny_linear_kernel<kTiles><<<grid, kLinearThreads, 0, stream>>>(
        static_cast<const uint16_t *>(a), static_cast<const uint16_t *>(w),
        static_cast<uint16_t *>(out), tokens, rows, cols);
    return static_cast<int32_t>(hipGetLastError());
}

// Tiles per workgroup: what spreads W's rows over one workgroup per CU, since
// each workgroup reads all of A (from L2): at 11008 x 4096 and 16 rows of A,
// 688 workgroups of one tile took 28 us, 230 of three 23.4 us.
constexpr int32_t kCus = 256;

// A launch has fewer than 2^32 threads; workgroups of the most tiles.
constexpr int64_t kMaxLinearRows = ((int64_t{1} << 32) / kLinearThreads - 1) * 4 * kTile;

}  // namespace
}  // namespace lct

using namespace lct;

extern "C" int32_t lct_skinny_linear(const void *a, const void *w, void *out, int32_t tokens,
                                     int32_t rows, int32_t cols, hipStream_t stream) {
    if (!a || !w || !out) return LCT_E_NULL;
    if (tokens <= 0 || tokens > LCT_MAX_SKINNY_TOKENS || rows <= 0 || cols <= 0
        || rows > kMaxLinearRows || cols > (1 << 30))
        return LCT_E_SIZE;
    if ((cols & 7) != 0
        || ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 15) != 0
        || (reinterpret_cast<uintptr_t>(out) & 1) != 0)
        return LCT_E_ARG;
    const int32_t tiles = ((rows + kTile - 1) / kTile + kCus - 1) / kCus;
    switch (tiles) {
    case 1: return launch_skinny<1>(a, w, out, tokens, rows, cols, stream);
    case 2: return launch_skinny<2>(a, w, out, tokens, rows, cols, stream);
    case 3: return launch_skinny<3>(a, w, out, tokens, rows, cols, stream);
    default: return launch_skinny<4>(a, w, out, tokens, rows, cols, stream);
    }
}
