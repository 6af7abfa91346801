// Decoder with fused overflow overlay (gfx950).
//
// Replaces LCT/kernels/generic/decode.py:174-308 (_decode_kernel and
// _decode_overflow_kernel).  One workgroup per codec block: stage the block's
// payload and tables in LDS, expand its overflow list, then every lane walks
// its stream two symbols per iteration, joining each exponent with its side
// byte and storing the BF16 bits at the swizzled logical offset.  Steps at or
// past a stream's overflow start take their exponent from the tail bytes and
// consume no payload bits.
//
// Three kernels share that work: the wide one described here, a compact one
// and a grouped one, which most grids take (choose_decoder); the latter two
// have their own comments.
//
// The step loop runs in 16-step chunks, each in two phases.  The decode
// phase walks the 16 steps using only LDS (payload, tables, overflow tails)
// and keeps the exponent fields in registers.  The store phase then waits for
// the chunk's side bytes, which were fetched one chunk earlier, issues the next
// chunk's fetch and writes the 16 BF16 values through a wave-private LDS tile
// as 16-byte stores (81.8 -> 78.2 us at 4096 blocks on gfx950 against 4-byte
// stores of lane pairs).  Each stream's first three payload words start in
// registers and only rows 3..W-1 are staged, which keeps the workgroup at
// 19.5 KiB of LDS with the tile; 64 VGPRs keep 8 waves per SIMD.  On gfx9 loads and stores share
// one counter, so a wait for a load also waits for every older store: with the
// decode phase between a chunk's stores and the next wait, those stores have
// drained by the time the wave waits.  The overflow check is only compiled into
// chunks that reach the wave's first overflow start.
#include <atomic>

#include "decode_core.h"

namespace lct {
namespace {

// Store phase of a full block.  The 8 rows' values go through a wave-private
// 1 KiB LDS tile (8 rows x the wave's 64 columns x 2 bytes) in column order,
// and each lane then stores 16 bytes (8 columns of one row): a wave store
// covers 8 whole 128-byte lines, where a direct store from the decoding lanes
// could only write 2 bytes (or 4, pairing lanes over DPP) per lane.  A wave's
// 64 lanes hold the 64 columns of one aligned group of a row: lane l of the
// wave holds column G + (l ^ (m & 63)) of group G = 64 * wave ^ (m & 192),
// m = the row's swizzle mask.  `first_step` and the block's first row are
// multiples of 8, so rows first_step + j and first_step + j + 1 (j even) share
// mask m0 ^ j, m0 = the mask of row first_step.
__device__ __forceinline__ void store_fields_tile(const uint32_t (&f)[kHalfSteps],
                                                  const uint8_t *slice, int slice_step,
                                                  uint16_t *tile, __amdgpu_buffer_rsrc_t out,
                                                  int first_step, int64_t row_base) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t m0 = static_cast<uint32_t>((row_base + first_step) & 254);
#pragma unroll
    for (int j = 0; j < kHalfSteps; j += 2) {
        const uint32_t pos = lane ^ ((m0 ^ static_cast<uint32_t>(j)) & (kWave - 1));
        tile[j * kWave + pos] =
            static_cast<uint16_t>(join_entry(f[j], side_byte(slice, slice_step + j)));
        tile[(j + 1) * kWave + pos] =
            static_cast<uint16_t>(join_entry(f[j + 1], side_byte(slice, slice_step + j + 1)));
    }
    // Lane l stores row r = first_step + (l >> 3), columns (l & 7) * 8.. of
    // the row's group.
    const uint4 q = reinterpret_cast<const uint4 *>(tile)[lane];
    const uint32_t r = lane >> 3;
    const uint32_t mask = m0 ^ (r & 6u);
    const uint32_t group = ((threadIdx.x & ~(kWave - 1u)) ^ (mask & 192u));
    const uint32_t offset = (group + (lane & 7u) * 8u) * 2u + r * (kLanes * 2u);
    store_b128<kStreaming>(q, out, offset + static_cast<uint32_t>(first_step) * (kLanes * 2));
}

// Store phase of the last, partial block: 2-byte stores of the positions
// inside the tensor.
__device__ __forceinline__ void store_fields_partial(const uint32_t (&f)[kHalfSteps],
                                                     const uint8_t *slice, int slice_step,
                                                     __amdgpu_buffer_rsrc_t out, int first_step,
                                                     int64_t row_base, uint32_t valid_in_block) {
    const uint32_t chunk_col2 = logical_col2(row_base, first_step);
#pragma unroll
    for (int j = 0; j < kHalfSteps; j += 2) {
        const int step = first_step + j;
        const uint32_t out0 = join_entry(f[j], side_byte(slice, slice_step + j));
        const uint32_t out1 = join_entry(f[j + 1], side_byte(slice, slice_step + j + 1));
        const int row_bytes = step * kLanes * 2;
        const uint32_t col2 = chunk_col2 ^ static_cast<uint32_t>(2 * j);
        const uint32_t off0 = static_cast<uint32_t>(step) * kLanes + (col2 >> 1);
        if (off0 < valid_in_block)
            __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(out0), out, col2,
                                                  row_bytes, kStreaming);
        if (off0 + kLanes < valid_in_block)
            __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(out1), out, col2,
                                                  row_bytes + kLanes * 2, kStreaming);
    }
}

template <bool kFull>
__device__ __forceinline__ void store_fields(const uint32_t (&f)[kHalfSteps], const uint8_t *slice,
                                             int slice_step, uint16_t *tile,
                                             __amdgpu_buffer_rsrc_t out, int first_step,
                                             int64_t row_base, uint32_t valid_in_block) {
    if (kFull)
        store_fields_tile(f, slice, slice_step, tile, out, first_step, row_base);
    else
        store_fields_partial(f, slice, slice_step, out, first_step, row_base, valid_in_block);
}

// Chunks [c_begin, c_end) with one overlay variant.  `side_next` holds the side
// bytes of chunk c_begin on entry and of chunk c_end on exit.
template <bool kFull, Overlay kOverlay, int S>
__device__ __forceinline__ void decode_chunks(StreamCursor &cursor, const LaneOverlay &lane,
                                              const uint8_t *tail_lds, uint8_t *slice,
                                              uint16_t *tile,
                                              __amdgpu_buffer_rsrc_t side, SideChunk &side_next,
                                              __amdgpu_buffer_rsrc_t out, int64_t row_base,
                                              uint32_t valid_in_block, int c_begin, int c_end) {
    const uint32_t voffset = side_fetch_offset();
#pragma unroll 1
    for (int c = c_begin; c < c_end; c += kChunkSteps) {
        uint32_t f[kHalfSteps];
        decode_fields<kFull, kOverlay>(cursor, lane, tail_lds, c, row_base, valid_in_block, f);
        store_side_chunk(slice, side_next);
        if (c + kChunkSteps < S) side_next = fetch_side_chunk(side, voffset, c + kChunkSteps);
        store_fields<kFull>(f, slice, 0, tile, out, c, row_base, valid_in_block);
        decode_fields<kFull, kOverlay>(cursor, lane, tail_lds, c + kHalfSteps, row_base,
                                       valid_in_block, f);
        store_fields<kFull>(f, slice, kHalfSteps, tile, out, c + kHalfSteps, row_base,
                            valid_in_block);
    }
}

// S is a template parameter so the chunk loops have fixed bounds.  Chunks that
// end at or before the wave's first overflow start skip the overlay check.
template <bool kFull, int S>
__device__ __forceinline__ void decode_rows(StreamCursor cursor, const LaneOverlay &lane,
                                            const uint8_t *tail_lds, uint8_t *slice,
                                            uint16_t *tile,
                                            __amdgpu_buffer_rsrc_t side, SideChunk side_next,
                                            __amdgpu_buffer_rsrc_t out, int64_t row_base,
                                            uint32_t valid_in_block) {
    static_assert(S % kChunkSteps == 0, "whole chunks");
    const int split = min(S, lane.wave_start & ~(kChunkSteps - 1));
    decode_chunks<kFull, kNoOverlay, S>(cursor, lane, tail_lds, slice, tile, side, side_next,
                                        out, row_base, valid_in_block, 0, split);
    if (split == S) return;
    if (lane.lds)
        decode_chunks<kFull, kLdsOverlay, S>(cursor, lane, tail_lds, slice, tile, side,
                                             side_next, out, row_base, valid_in_block, split, S);
    else
        decode_chunks<kFull, kHbmOverlay, S>(cursor, lane, tail_lds, slice, tile, side,
                                             side_next, out, row_base, valid_in_block, split, S);
}

// 8 waves per SIMD: the compiler keeps to 64 VGPRs (65 unconstrained).
// Codec block `block` of one tensor, by the workgroup.
__device__ __forceinline__ void decode_block_wide(
    const int32_t *__restrict__ encoded, const uint8_t *__restrict__ side,
    uint16_t *__restrict__ output, const int32_t *__restrict__ shifted_decode,
    const int32_t *__restrict__ center_ptr, int64_t n_blocks, int64_t logical_numel, int S,
    int W, int rare, const lct_overflow &ov, int has_overlay, int64_t block) {
    extern __shared__ uint32_t stage[];   // register_stage_bytes(W): rows 3..W-1
    __shared__ DecodeTables tb;
    __shared__ int32_t scratch[kWavesPerBlock];
    __shared__ uint8_t tail_lds[kTailLds];
    __shared__ __attribute__((aligned(16))) uint16_t out_tiles[kWavesPerBlock][kHalfSteps * kWave];
    // The overflow maps (2 KiB) are only used before the first side chunk is
    // stored, so they share the side slices' LDS.
    __shared__ __attribute__((aligned(16))) uint8_t side_slices[kWavesPerBlock][kChunkSteps * kWave];
    int32_t *map_start = reinterpret_cast<int32_t *>(&side_slices[0][0]);
    int32_t *map_offset = map_start + kLanes;
    const int64_t row_base = block * S;
    const int64_t logical_base = row_base * kLanes;
    const uint32_t block_elems = static_cast<uint32_t>(S) * kLanes;
    const int64_t remaining = logical_numel - logical_base;
    const uint32_t valid = remaining < block_elems ? static_cast<uint32_t>(remaining) : block_elems;
    const __amdgpu_buffer_rsrc_t side_rsrc = make_rsrc(side + logical_base, block_elems);
    const __amdgpu_buffer_rsrc_t out_rsrc = make_rsrc(output + logical_base, 2u * valid);
    // The first side chunk is in flight while the prologue stages the payload.
    const SideChunk first = fetch_side_chunk(side_rsrc, side_fetch_offset(), 0);

    uint32_t words[kRegisterRows];
    load_register_rows(encoded, n_blocks * kLanes, block, words);

    const int32_t center = center_ptr[0];
    build_decode_tables(tb, shifted_decode, center);
    stage_payload_rows(stage, encoded, n_blocks * kLanes, block, kRegisterRows, W);
    const LaneOverlay lane = build_overlay(ov, has_overlay != 0, block, n_blocks, S, map_start,
                                           map_offset, scratch, tail_lds, kTailLds);
    wait_memory();
    __syncthreads();   // payload and tails visible; overflow maps no longer read

    StreamCursor cursor;
    cursor.init_registers(stage + threadIdx.x, &tb, static_cast<uint32_t>(W), rare, words[0],
                          words[1], words[2]);
    uint8_t *slice = side_slices[threadIdx.x / kWave];
    uint16_t *tile = out_tiles[threadIdx.x / kWave];
    if (valid == block_elems) {
        if (S == 128)
            decode_rows<true, 128>(cursor, lane, tail_lds, slice, tile, side_rsrc, first,
                                   out_rsrc, row_base, valid);
        else
            decode_rows<true, 256>(cursor, lane, tail_lds, slice, tile, side_rsrc, first,
                                   out_rsrc, row_base, valid);
    } else {
        if (S == 128)
            decode_rows<false, 128>(cursor, lane, tail_lds, slice, tile, side_rsrc, first,
                                    out_rsrc, row_base, valid);
        else
            decode_rows<false, 256>(cursor, lane, tail_lds, slice, tile, side_rsrc, first,
                                    out_rsrc, row_base, valid);
    }
}

__global__ __launch_bounds__(kLanes, 8) void decode_kernel(
    const int32_t *__restrict__ encoded, const uint8_t *__restrict__ side,
    uint16_t *__restrict__ output, const int32_t *__restrict__ shifted_decode,
    const int32_t *__restrict__ center_ptr, int64_t n_blocks, int64_t logical_numel, int S,
    int W, int rare, lct_overflow ov, int has_overlay) {
    decode_block_wide(encoded, side, output, shifted_decode, center_ptr, n_blocks, logical_numel,
                      S, W, rare, ov, has_overlay, blockIdx.x);
}

// Several tensors in one launch (LCT_MAX_DECODE_BATCH at most): workgroup b
// decodes block b - first_block[j] of job j, the last job whose first block
// is at most b.  For tensors of a few codec blocks each (a layer's weights),
// whose decodes are bound by one block's latency, one launch replaces one per
// tensor.  The job table travels in the kernel arguments.
struct DecodeBatchJob {
    const int32_t *encoded;
    const uint8_t *side;
    uint16_t *output;
    const int32_t *shifted_decode;
    const int32_t *center;
    int64_t n_blocks;
    int64_t logical_numel;
    int32_t steps;
    int32_t fixed_words;
    int32_t rare;
    int32_t has_overlay;
    lct_overflow ov;
};

struct DecodeBatch {
    int32_t n_jobs;
    int32_t first_block[LCT_MAX_DECODE_BATCH + 1];
    DecodeBatchJob jobs[LCT_MAX_DECODE_BATCH];
};

__device__ __forceinline__ int batch_job(const DecodeBatch &batch, int32_t b) {
    int j = 0;
    for (int k = 1; k < batch.n_jobs; ++k)
        if (b >= batch.first_block[k]) j = k;
    return j;
}

__global__ __launch_bounds__(kLanes, 8) void decode_batch_kernel(DecodeBatch batch) {
    const int32_t b = static_cast<int32_t>(blockIdx.x);
    const int j = batch_job(batch, b);
    const DecodeBatchJob &job = batch.jobs[j];
    decode_block_wide(job.encoded, job.side, job.output, job.shifted_decode, job.center,
                      job.n_blocks, job.logical_numel, job.steps, job.fixed_words, job.rare,
                      job.ov, job.has_overlay, b - batch.first_block[j]);
}

// ---- the compact decoder: 8 workgroups per CU for payloads of 13 to 19 words
//
// The kernel above keeps 10 KiB of LDS beside its payload stage (the tables,
// the tails, a 1 KiB side slice and a 1 KiB output tile per wave), so from
// W = 13 on it holds more than 20 KiB and fewer than 8 workgroups fit on a CU
// (C2's W = 19: 26 KiB, 6 per CU, so 2048 blocks ran in 1.33 rounds).  This
// variant keeps 3.5 KiB beside the stage (19.5 KiB at W = 19):
//  * side bytes move in 8-step halves, 8 bytes per lane, through a 512-byte
//    region per wave, which then also serves as a 4-row output tile: a lane
//    reads its 8 side bytes before any lane writes the tile (a wave's LDS
//    accesses complete in program order), and each 4-row tile leaves with one
//    8-byte store per lane (4 whole 128-byte lines per wave store);
//  * the escape table is not kept: an escaped literal's exponent field is
//    computed from the center (escapes are rare and take a wave-uniform
//    branch);
//  * the overflow maps (2 KiB) share the four regions before the first half.
// Side bytes are fetched two halves (one 16-step chunk) ahead, as above.

struct CompactDecodeTables {
    uint16_t entry[256];

    __device__ __forceinline__ uint32_t escaped(uint32_t literal, int32_t center) const {
        return static_cast<uint32_t>(
                   (index_to_exponent(static_cast<int32_t>(literal), center) + 127) & 255)
            << 7;
    }
    static __device__ __forceinline__ uint32_t tail(uint32_t byte) {
        return DecodeTables::tail(byte);
    }
};

using CompactCursor = StreamCursorT<kLanes, CompactDecodeTables>;

constexpr int kRegionBytes = kHalfSteps * kWave;   // 512: 8 side rows, or a 4-row tile

// Buffer offset of this lane's 8 bytes within an 8-step half: row j >> 3,
// columns (j & 7) * 8 .. + 8 of the wave's 64-column segment.
__device__ __forceinline__ uint32_t side_half_offset() {
    const uint32_t j = threadIdx.x & (kWave - 1);
    return (j >> 3) * kLanes + (threadIdx.x / kWave) * kWave + (j & 7) * 8;
}

__device__ __forceinline__ uint2 fetch_side_half(__amdgpu_buffer_rsrc_t side, uint32_t voffset,
                                                 int first_step) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(
                                         side, voffset, first_step * kLanes, 0));
}

// The half's entries f joined with its side bytes (q: this lane's 8 fetched
// bytes), stored at their logical positions: full blocks through two 4-row
// tiles in `region`, the last block with 2-byte stores of the positions
// inside the tensor.
template <bool kFull>
__device__ __forceinline__ void store_half_compact(const uint32_t (&f)[kHalfSteps], uint2 q,
                                                   uint8_t *region, __amdgpu_buffer_rsrc_t out,
                                                   int first_step, int64_t row_base,
                                                   uint32_t valid_in_block) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    reinterpret_cast<uint2 *>(region)[lane] = q;   // byte s * 64 + column: step s
    uint32_t v[kHalfSteps];
#pragma unroll
    for (int j = 0; j < kHalfSteps; ++j) v[j] = join_entry(f[j], region[j * kWave + lane]);
    if (!kFull) {
        const uint32_t chunk_col2 = logical_col2(row_base, first_step);
#pragma unroll
        for (int j = 0; j < kHalfSteps; j += 2) {
            const int step = first_step + j;
            const int row_bytes = step * kLanes * 2;
            const uint32_t col2 = chunk_col2 ^ static_cast<uint32_t>(2 * j);
            const uint32_t off0 = static_cast<uint32_t>(step) * kLanes + (col2 >> 1);
            if (off0 < valid_in_block)
                __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(v[j]), out, col2,
                                                      row_bytes, kStreaming);
            if (off0 + kLanes < valid_in_block)
                __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(v[j + 1]), out, col2,
                                                      row_bytes + kLanes * 2, kStreaming);
        }
        return;
    }
    // Tile rows r = 0..3 hold half rows 4t + r; lane l of the wave holds
    // column l ^ (m & 63) of the row's group (m: the row's swizzle mask), and
    // then stores 8 bytes: columns (l & 15) * 4 .. + 4 of tile row l >> 4.
    // first_step and the block's first row are multiples of 8, so half row r
    // has mask m0 ^ (r & 6).
    uint16_t *tile = reinterpret_cast<uint16_t *>(region);
    const uint32_t m0 = static_cast<uint32_t>((row_base + first_step) & 254);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t row = static_cast<uint32_t>(4 * t + r);
            tile[r * kWave + (lane ^ ((m0 ^ (row & 6u)) & (kWave - 1)))] =
                static_cast<uint16_t>(v[4 * t + r]);
        }
        const uint2 d = reinterpret_cast<const uint2 *>(tile)[lane];
        const uint32_t row = 4u * t + (lane >> 4);
        const uint32_t mask = m0 ^ (row & 6u);
        const uint32_t group = (threadIdx.x & ~(kWave - 1u)) ^ (mask & 192u);
        const uint32_t offset = (group + (lane & 15u) * 4u) * 2u
            + (static_cast<uint32_t>(first_step) + row) * (kLanes * 2u);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(
                                                  __attribute__((ext_vector_type(2))) uint32_t, d),
                                              out, offset, 0, kStreaming);
    }
}

// Halves [h_begin, h_end) (in steps) with one overlay variant.  On entry
// `ahead0` and `ahead1` hold the side bytes of halves h_begin and h_begin + 8;
// on exit those of h_end and h_end + 8.
template <bool kFull, Overlay kOverlay, int S>
__device__ __forceinline__ void decode_halves_compact(CompactCursor &cursor,
                                                      const LaneOverlay &lane,
                                                      const uint8_t *tail_lds, uint8_t *region,
                                                      __amdgpu_buffer_rsrc_t side, uint2 &ahead0,
                                                      uint2 &ahead1, __amdgpu_buffer_rsrc_t out,
                                                      int64_t row_base, uint32_t valid_in_block,
                                                      int h_begin, int h_end) {
    const uint32_t voffset = side_half_offset();
#pragma unroll 1
    for (int h = h_begin; h < h_end; h += kHalfSteps) {
        uint32_t f[kHalfSteps];
        decode_fields<kFull, kOverlay>(cursor, lane, tail_lds, h, row_base, valid_in_block, f);
        const uint2 q = ahead0;
        ahead0 = ahead1;
        if (h + 2 * kHalfSteps < S)
            ahead1 = fetch_side_half(side, voffset, h + 2 * kHalfSteps);
        store_half_compact<kFull>(f, q, region, out, h, row_base, valid_in_block);
    }
}

template <bool kFull, int S>
__device__ __forceinline__ void decode_rows_compact(CompactCursor cursor, const LaneOverlay &lane,
                                                    const uint8_t *tail_lds, uint8_t *region,
                                                    __amdgpu_buffer_rsrc_t side, uint2 ahead0,
                                                    uint2 ahead1, __amdgpu_buffer_rsrc_t out,
                                                    int64_t row_base, uint32_t valid_in_block) {
    const int split = min(S, lane.wave_start & ~(kHalfSteps - 1));
    decode_halves_compact<kFull, kNoOverlay, S>(cursor, lane, tail_lds, region, side, ahead0,
                                                ahead1, out, row_base, valid_in_block, 0, split);
    if (split == S) return;
    if (lane.lds)
        decode_halves_compact<kFull, kLdsOverlay, S>(cursor, lane, tail_lds, region, side,
                                                     ahead0, ahead1, out, row_base,
                                                     valid_in_block, split, S);
    else
        decode_halves_compact<kFull, kHbmOverlay, S>(cursor, lane, tail_lds, region, side,
                                                     ahead0, ahead1, out, row_base,
                                                     valid_in_block, split, S);
}

// LDS beside the payload stage: the entry table, scan scratch, the tails and
// the four regions.
constexpr int32_t kCompactStaticLds = 512 + 16 + kTailLds + kWavesPerBlock * kRegionBytes;
static_assert(register_stage_bytes(19) + kCompactStaticLds <= 20 * 1024,
              "MEDIUM's payload (W = 19) keeps 8 workgroups per CU");

__global__ __launch_bounds__(kLanes, 8) void decode_kernel_compact(
    const int32_t *__restrict__ encoded, const uint8_t *__restrict__ side,
    uint16_t *__restrict__ output, const int32_t *__restrict__ shifted_decode,
    const int32_t *__restrict__ center_ptr, int64_t n_blocks, int64_t logical_numel, int S,
    int W, int rare, lct_overflow ov, int has_overlay) {
    extern __shared__ uint32_t stage[];   // register_stage_bytes(W): rows 3..W-1
    __shared__ CompactDecodeTables tb;
    __shared__ int32_t scratch[kWavesPerBlock];
    __shared__ uint8_t tail_lds[kTailLds];
    __shared__ __attribute__((aligned(16))) uint8_t regions[kWavesPerBlock][kRegionBytes];
    static_assert(sizeof(regions) >= 2 * kLanes * sizeof(int32_t), "the overflow maps fit");
    int32_t *map_start = reinterpret_cast<int32_t *>(&regions[0][0]);
    int32_t *map_offset = map_start + kLanes;
    const int64_t block = blockIdx.x;
    const int64_t row_base = block * S;
    const int64_t logical_base = row_base * kLanes;
    const uint32_t block_elems = static_cast<uint32_t>(S) * kLanes;
    const int64_t remaining = logical_numel - logical_base;
    const uint32_t valid = remaining < block_elems ? static_cast<uint32_t>(remaining) : block_elems;
    const __amdgpu_buffer_rsrc_t side_rsrc = make_rsrc(side + logical_base, block_elems);
    const __amdgpu_buffer_rsrc_t out_rsrc = make_rsrc(output + logical_base, 2u * valid);
    // The first two side halves are in flight while the prologue stages the
    // payload.
    const uint32_t voffset = side_half_offset();
    const uint2 ahead0 = fetch_side_half(side_rsrc, voffset, 0);
    const uint2 ahead1 = fetch_side_half(side_rsrc, voffset, kHalfSteps);

    uint32_t words[kRegisterRows];
    load_register_rows(encoded, n_blocks * kLanes, block, words);

    const int32_t center = center_ptr[0];
    {
        const int32_t packed = shifted_decode[threadIdx.x];
        const int32_t length = packed & 255;
        const uint32_t field = static_cast<uint32_t>(((packed >> 8) + 127) & 255) << 7;
        tb.entry[threadIdx.x] = static_cast<uint16_t>(
            (length >= 1 && length <= 8) ? (static_cast<uint32_t>(length) | field)
                                         : static_cast<uint32_t>(kEscapeLength));
    }
    stage_payload_rows(stage, encoded, n_blocks * kLanes, block, kRegisterRows, W);
    const LaneOverlay lane = build_overlay(ov, has_overlay != 0, block, n_blocks, S, map_start,
                                           map_offset, scratch, tail_lds, kTailLds);
    wait_memory();
    __syncthreads();   // payload and tails visible; overflow maps no longer read

    CompactCursor cursor;
    cursor.init_registers(stage + threadIdx.x, &tb, static_cast<uint32_t>(W), rare, words[0],
                          words[1], words[2], center);
    uint8_t *region = regions[threadIdx.x / kWave];
    if (valid == block_elems) {
        if (S == 128)
            decode_rows_compact<true, 128>(cursor, lane, tail_lds, region, side_rsrc, ahead0,
                                           ahead1, out_rsrc, row_base, valid);
        else
            decode_rows_compact<true, 256>(cursor, lane, tail_lds, region, side_rsrc, ahead0,
                                           ahead1, out_rsrc, row_base, valid);
    } else {
        if (S == 128)
            decode_rows_compact<false, 128>(cursor, lane, tail_lds, region, side_rsrc, ahead0,
                                            ahead1, out_rsrc, row_base, valid);
        else
            decode_rows_compact<false, 256>(cursor, lane, tail_lds, region, side_rsrc, ahead0,
                                            ahead1, out_rsrc, row_base, valid);
    }
}

// ---- the grouped decoder: several symbols per table lookup
//
// The kernels above take two dependent LDS lookups per symbol pair, so a
// stream of 256 symbols is a chain of 256 lookups: with a few workgroups per
// CU (a layer's weights, one activation) that chain is the launch's time, not
// HBM.  Here one lookup of 10 bits gives up to four whole symbols (3.2 to 3.4
// on the codebooks' own data), three lookups are taken from each 32-bit
// window, and the exponent bytes go to an LDS tile of rows instead of staying
// in registers in lock step, so lanes may run ahead of one another:
//  * a wave decodes its 64 streams until each has kTileSteps more rows (or is
//    at its end: its first overflow step, or the tensor's end), every lane at
//    its own pace; a lookup's four exponent bytes are stored at the lane's
//    next four rows, and those past its symbol count are overwritten later;
//  * rows at and past a stream's overflow start are then filled from its tail;
//  * the wave joins the tile's rows with their side bytes, fetched one tile
//    ahead: lane j takes 8 columns of the four rows 4 (8 u + (j >> 3)) + i of
//    each 32-row unit u, so a 16-byte read of the tile holds four columns of
//    all four rows, the swizzle's XOR by i is a change of the output's words
//    and every wave store is 8 whole 128-byte lines;
//  * rows already decoded past the tile's end move to its start.
// The tensor's last, partial block differs only in its streams' ends and in
// the stores of the piece that holds the tensor's end.
//
// What bounds it: with up to one workgroup per CU the chain of lookups (27 turns
// of three per 256 symbols; 15.6 us per public decompress at 36 blocks of 256
// steps against the wide kernel's 24.4), then the LDS (22.5 us at 512 blocks),
// from about 688 blocks on HBM (28.1 us, 5.4 TB/s; 86.2 us at 4096 blocks of
// 128 steps against 89.4).  Measured against an earlier form (28.8 us at 688): the exponent bytes stored one by one in row-major tiles
// (12 byte stores per turn: 29.6 against 28.8 us at 688 blocks, 23.2 at 512);
// 9-bit tables or 32-row tiles (more workgroups per CU, but 15.3 to 17.7 us at
// 36 blocks and 0.4 to 2 us slower at 4096).
constexpr int kGroupBits = 10;      // table index bits: three lookups fit a 32-bit window
constexpr int kGroupLookups = 3;
constexpr int kGroupSymbols = 4;    // symbols per entry at most
constexpr int kTileSteps = 64;
constexpr int kUnits = kTileSteps / 32;
// A lane passes its target by at most 3 lookups of 4 symbols less one.
constexpr int kTileSpare = kGroupLookups * kGroupSymbols;
// The tile holds dwords of four rows of one lane, the 64 lanes' dwords of a
// row quad side by side, so lanes at different rows still hit 64 banks.
constexpr int kQuadBytes = kWave * 4;
constexpr int kTileBytes = (kTileSteps + kTileSpare + 4) / 4 * kQuadBytes;   // one wave's

// Entries {up to 4 exponent bytes, total length | symbols * 8 << 8}; y = 0
// where the first symbol is an escape.
struct GroupTables {
    uint2 entry[1 << kGroupBits];
};

// From the 1024-entry shifted decode table's first 256 entries: `base` (LDS,
// 256 dwords) holds length | exponent << 8, 0 for an escape or a code longer
// than 8 bits.  Bits past the index read as 0: a symbol is taken only if its
// code ends within the index, and then those bits had no part in it.
__device__ __forceinline__ void build_group_tables(GroupTables &tb, uint32_t *base,
                                                   int32_t packed) {
    const int t = threadIdx.x;
    const int32_t length = packed & 255;
    const uint32_t exponent = static_cast<uint32_t>((packed >> 8) + 127) & 255u;
    base[t] = length >= 1 && length <= 8 ? static_cast<uint32_t>(length) | (exponent << 8) : 0u;
    __syncthreads();
    constexpr int kPer = (1 << kGroupBits) / kLanes;
    uint32_t at[kPer], bytes[kPer], count[kPer];
    bool open[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        at[k] = bytes[k] = count[k] = 0u;
        open[k] = true;
    }
#pragma unroll
    for (int s = 0; s < kGroupSymbols; ++s) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const uint32_t index = static_cast<uint32_t>(t + k * kLanes);
            const uint32_t b = base[(index >> at[k]) & 255u];
            const uint32_t end = at[k] + (b & 255u);
            open[k] = open[k] && b != 0u && end <= static_cast<uint32_t>(kGroupBits);
            if (open[k]) {
                bytes[k] |= (b >> 8) << (8 * s);
                count[k] += 1u;
                at[k] = end;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k)
        tb.entry[t + k * kLanes] = make_uint2(bytes[k], at[k] | (count[k] * 8u) << 8);
}

// The tile is written by dword and by byte and read 16 bytes at a time: types
// that may alias each other.
using TileDword = __attribute__((may_alias)) uint32_t;
typedef uint32_t TileDwords __attribute__((ext_vector_type(4), may_alias));

// One lane's column of the tile, filled from the top: `row8` is 8 x the next
// row and `word` the rows of its dword so far.
struct TileColumn {
    uint8_t *base;
    uint32_t row8, word;

    // Append a lookup's exponent bytes (the bytes past its symbols are 0);
    // advance8 = 8 x their number.  Every append stores the dword it began in;
    // one that also fills it leaves the rest in the next.
    __device__ __forceinline__ void append(uint32_t bytes, uint32_t advance8) {
        const uint64_t placed = static_cast<uint64_t>(bytes) << (row8 & 24u);
        const uint32_t first = word | static_cast<uint32_t>(placed);
        *dword() = first;
        const uint32_t next8 = row8 + advance8;
        word = (next8 ^ row8) >= 32u ? static_cast<uint32_t>(placed >> 32) : first;
        row8 = next8;
    }

    // Store the dword being filled (after a tile's last append).
    __device__ __forceinline__ void flush() const { *dword() = word; }

    __device__ __forceinline__ TileDword *dword() const {
        return reinterpret_cast<TileDword *>(base + (row8 & ~31u) * (kQuadBytes / 32));
    }
};

// Two BF16 values from their exponent bytes (bytes 2p, 2p + 1 of e) and side
// bytes (of sm): each half becomes exponent << 8 | side, whose exponent moves
// down one bit and whose sign moves up to bit 15.
template <int kHalf>
__device__ __forceinline__ uint32_t join_two(uint32_t e, uint32_t sm) {
    const uint32_t x = __builtin_amdgcn_perm(e, sm, kHalf == 0 ? 0x05010400u : 0x07030602u);
    uint32_t low, out;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(low) : "s"(0x007F007Fu), "v"(x), "v"(x << 8));
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(out) : "s"(0x7F807F80u), "v"(x >> 1), "v"(low));
    return out;
}

// Byte k of the four words of `w`, for k = 0..3: rows of a 4 x 4 byte block
// whose columns are the words.
__device__ __forceinline__ void transpose_bytes(TileDwords w, uint32_t &r0, uint32_t &r1, uint32_t &r2,
                                                uint32_t &r3) {
    // v_perm_b32(s0, s1, sel): bytes 0..3 select s1, 4..7 s0.
    const uint32_t a01 = __builtin_amdgcn_perm(w.y, w.x, 0x05010400u);   // x0 y0 x1 y1
    const uint32_t b01 = __builtin_amdgcn_perm(w.w, w.z, 0x05010400u);
    const uint32_t a23 = __builtin_amdgcn_perm(w.y, w.x, 0x07030602u);   // x2 y2 x3 y3
    const uint32_t b23 = __builtin_amdgcn_perm(w.w, w.z, 0x07030602u);
    r0 = __builtin_amdgcn_perm(b01, a01, 0x05040100u);
    r1 = __builtin_amdgcn_perm(b01, a01, 0x07060302u);
    r2 = __builtin_amdgcn_perm(b23, a23, 0x05040100u);
    r3 = __builtin_amdgcn_perm(b23, a23, 0x07060302u);
}

// Of a tile, lane j takes the 4 rows of quad 8 u + (j >> 3) and 8 columns,
// for each u: kUnits units of 4 rows x 8 columns.
struct GroupSides {
    uint2 q[kUnits][4];
};

// Offset of thread `thread`'s first unit within a row of the block's side
// bytes; out of range for a tile past the block's last (the fetch one tile
// ahead of the last one).
constexpr uint32_t group_side_offset(uint32_t thread, int first_step, int S) {
    const uint32_t j = thread & (kWave - 1);
    return first_step < S ? (j >> 3) * (4 * kLanes) + (thread & ~(kWave - 1u)) + (j & 7) * 8
                          : kOutOfRange;
}

// Whether every fetch of a block, the one past its end among them, reads
// inside its S rows or is out of range by its VGPR offset alone.
constexpr bool group_sides_in_block(int S) {
    for (int first = 0; first <= S; first += kTileSteps)
        for (uint32_t thread = 0; thread < kLanes; ++thread) {
            const uint32_t offset = group_side_offset(thread, first, S);
            const uint32_t last = static_cast<uint32_t>(first + 32 * (kUnits - 1) + 3) * kLanes;
            if (offset != kOutOfRange && offset + last + 8 > static_cast<uint32_t>(S) * kLanes)
                return false;
        }
    return true;
}
static_assert(group_sides_in_block(128) && group_sides_in_block(256),
              "the side bytes' prefetch stays inside the block");

// The side bytes of this lane's units of the tile at `first_step` (0 past the
// block's end).
__device__ __forceinline__ void fetch_group_sides(GroupSides &s, __amdgpu_buffer_rsrc_t side,
                                                  int first_step, int S) {
    const uint32_t voffset = group_side_offset(threadIdx.x, first_step, S);
#pragma unroll
    for (int u = 0; u < kUnits; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            s.q[u][i] = __builtin_bit_cast(
                uint2, __builtin_amdgcn_raw_buffer_load_b64(
                           side, voffset, (first_step + 32 * u + i) * kLanes, 0));
}

// The tile's rows joined with their side bytes and stored.  Row r of the block
// has swizzle mask m = (row_base + r) & 254: lane 8 q + k of the wave holds
// column 8 (q ^ (m >> 3 & 7)) + (k ^ (m & 6)) of its 64-column group.  In
// row 4 R + i of the tile m & 4 is that of R, odd for half of the lanes (their
// two 4-lane halves change places), and m & 2 that of i.
__device__ __forceinline__ void store_tile(const uint8_t *tile, const GroupSides &s,
                                           __amdgpu_buffer_rsrc_t out, int first_step,
                                           int64_t row_base, bool full, uint32_t valid) {
    const uint32_t j = threadIdx.x & (kWave - 1);
    const uint32_t a = j >> 3, q = j & 7u;
    const bool swap = (a & 1u) != 0;
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
        const uint32_t row = static_cast<uint32_t>(first_step + 32 * u) + 4u * a;
        const uint32_t m = static_cast<uint32_t>(row_base + row) & 254u;
        const uint32_t column = ((threadIdx.x & ~(kWave - 1u)) ^ (m & 192u))
            + 8u * (q ^ ((m >> 3) & 7u));
        const uint8_t *quads = tile + (8 * u + a) * kQuadBytes + 32 * q;
        const TileDwords left = *reinterpret_cast<const TileDwords *>(quads + (swap ? 16 : 0));
        const TileDwords right = *reinterpret_cast<const TileDwords *>(quads + (swap ? 0 : 16));
        uint32_t el[4], er[4];
        transpose_bytes(left, el[0], el[1], el[2], el[3]);
        transpose_bytes(right, er[0], er[1], er[2], er[3]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t sl = swap ? s.q[u][i].y : s.q[u][i].x;
            const uint32_t sr = swap ? s.q[u][i].x : s.q[u][i].y;
            const uint32_t y[4] = {join_two<0>(el[i], sl), join_two<1>(el[i], sl),
                                   join_two<0>(er[i], sr), join_two<1>(er[i], sr)};
            const int x = i >> 1;
            const uint4 v = make_uint4(y[0 ^ x], y[1 ^ x], y[2 ^ x], y[3 ^ x]);
            const uint32_t element = (row + i) * kLanes + column;
            if (full || element + 8 <= valid) {
                store_b128<kStreaming>(v, out, element * 2u);
            } else if (element < valid) {
                const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k)
                    if (element + k < valid)
                        __builtin_amdgcn_raw_buffer_store_b16(
                            static_cast<uint16_t>(w[k / 2] >> (16 * (k & 1))), out,
                            (element + k) * 2u, 0, kStreaming);
            }
        }
    }
}

// An escape (y = 0) at bit `offset` (low 5 bits, at most 16) of `bits` becomes one
// symbol of at most 16 bits: ESC + 8-bit literal table index (primitives.py:
// 29-35).  A third lookup's window would then pass the 32 bits' end.
__device__ __forceinline__ void take_escape(uint2 &entry, uint32_t &third, uint32_t bits,
                                            uint32_t offset, int rare, int32_t center) {
    const bool escaped = entry.y == 0u;
    const uint32_t literal = __builtin_amdgcn_ubfe(bits, (offset & 31u) + rare, 8);
    const uint32_t exponent = static_cast<uint32_t>(
        index_to_exponent(static_cast<int32_t>(literal), center) + 127) & 255u;
    entry.x = escaped ? exponent : entry.x;
    entry.y = escaped ? static_cast<uint32_t>(rare + 8) | 8u << 8 : entry.y;
    third = escaped ? 0u : third;
}

// Codec block `block` of one tensor, by the workgroup.
__device__ __forceinline__ void decode_block_grouped(
    const int32_t *__restrict__ encoded, const uint8_t *__restrict__ side,
    uint16_t *__restrict__ output, const int32_t *__restrict__ shifted_decode,
    const int32_t *__restrict__ center_ptr, int64_t n_blocks, int64_t logical_numel, int S,
    int W, int rare, const lct_overflow &ov, int has_overlay, int64_t block) {
    extern __shared__ uint32_t stage[];   // register_stage_bytes(W): rows 3..W-1
    __shared__ __attribute__((aligned(16))) GroupTables tb;
    __shared__ int32_t scratch[kWavesPerBlock];
    __shared__ uint8_t tail_lds[kTailLds];
    __shared__ __attribute__((aligned(16))) uint8_t tiles[kWavesPerBlock][kTileBytes];
    // The base table and the overflow maps (3 KiB) are only used before the
    // first tile is decoded.
    uint32_t *base = reinterpret_cast<uint32_t *>(&tiles[0][0]);
    int32_t *map_start = reinterpret_cast<int32_t *>(base + kLanes);
    int32_t *map_offset = map_start + kLanes;
    const int t = threadIdx.x;
    const int64_t row_base = block * S;
    const int64_t logical_base = row_base * kLanes;
    const uint32_t block_elems = static_cast<uint32_t>(S) * kLanes;
    const int64_t remaining = logical_numel - logical_base;
    const uint32_t valid = remaining < block_elems ? static_cast<uint32_t>(remaining) : block_elems;
    const bool full = valid == block_elems;
    const __amdgpu_buffer_rsrc_t side_rsrc = make_rsrc(side + logical_base, block_elems);
    const __amdgpu_buffer_rsrc_t out_rsrc = make_rsrc(output + logical_base, 2u * valid);

    const int32_t packed = shifted_decode[t];
    const int32_t center = center_ptr[0];
    uint32_t words[kRegisterRows];
    load_register_rows(encoded, n_blocks * kLanes, block, words);
    stage_payload_rows(stage, encoded, n_blocks * kLanes, block, kRegisterRows, W);
    const OverlayHead head = load_overlay_head(ov, has_overlay != 0, block, n_blocks);
    GroupSides sides;
    fetch_group_sides(sides, side_rsrc, 0, S);
    build_group_tables(tb, base, packed);
    const LaneOverlay lane = build_overlay(ov, head, S, map_start, map_offset, scratch, tail_lds,
                                           kTailLds);
    wait_memory();
    __syncthreads();   // payload, table and tails visible; the maps no longer read

    // This stream's symbols in the payload: the rows before its overflow start
    // that lie inside the tensor.
    int32_t limit = lane.start;
    if (!full) {
        const int32_t rows = static_cast<int32_t>(valid / kLanes);
        const uint32_t column = static_cast<uint32_t>(t)
            ^ static_cast<uint32_t>((row_base + rows) & 254);
        limit = min(limit, rows + (column < valid % kLanes ? 1 : 0));
    }

    uint8_t *const tile = tiles[t / kWave];
    TileColumn column{tile + (t & (kWave - 1)) * 4, 0u, 0u};
    const uint32_t *const stage_lane = stage + t - kRegisterRows * kLanes;
    const uint32_t pad_row = static_cast<uint32_t>(W) - 1u;
    uint32_t lo = words[0], hi = words[1], nx = words[2], pos = 0, next_row = kRegisterRows;
#pragma unroll 1
    for (int first = 0; first < S; first += kTileSteps) {
        const int32_t target8 = 8 * min(kTileSteps, limit - first);   // may be negative
        if (static_cast<int32_t>(column.row8) < target8) {
            // Each lookup's bytes are appended while the next lookup is in
            // flight (the loop's last, e2's, in the next turn).
            uint32_t held = 0u, held8 = 0u, row8 = column.row8;
            do {
                const uint32_t pending = stage_lane[next_row * kLanes];
                const uint32_t bits = __builtin_amdgcn_alignbit(hi, lo, pos);
                uint2 e0 = tb.entry[bits & ((1u << kGroupBits) - 1u)];
                __builtin_amdgcn_sched_barrier(0);
                column.append(held, held8);
                __builtin_amdgcn_sched_barrier(0);
                uint32_t two;
                uint2 e2;
                if (__builtin_expect(__any(e0.y == 0u), 0)) {
                    // A turn of its own, which takes the second lookup's escape
                    // too: escapes come in runs, a row of larger values lying
                    // 30 steps long in every stream (a 2282 x 7616 tensor of
                    // such rows, 531 blocks of W = 22: 23.0 us with one escape
                    // per turn, 20.4 with two, the wide kernel 21.3; without
                    // escapes the same within 2 %).
                    uint32_t third = ~0u;
                    take_escape(e0, third, bits, 0u, rare, center);
                    uint2 e1 = tb.entry[__builtin_amdgcn_ubfe(bits, e0.y, kGroupBits)];
                    __builtin_amdgcn_sched_barrier(0);
                    column.append(e0.x, e0.y >> 8);
                    __builtin_amdgcn_sched_barrier(0);
                    take_escape(e1, third, bits, e0.y, rare, center);
                    two = e0.y + e1.y;
                    e2 = tb.entry[__builtin_amdgcn_ubfe(bits, two, kGroupBits)];
                    __builtin_amdgcn_sched_barrier(0);
                    column.append(e1.x, e1.y >> 8);
                    __builtin_amdgcn_sched_barrier(0);
                    e2.x &= third;
                    e2.y &= third;
                } else {
                    const uint2 e1 = tb.entry[__builtin_amdgcn_ubfe(bits, e0.y, kGroupBits)];
                    __builtin_amdgcn_sched_barrier(0);
                    column.append(e0.x, e0.y >> 8);
                    __builtin_amdgcn_sched_barrier(0);
                    two = e0.y + e1.y;   // lengths in bits 0..5, rows from bit 8
                    e2 = tb.entry[__builtin_amdgcn_ubfe(bits, two, kGroupBits)];
                    __builtin_amdgcn_sched_barrier(0);
                    column.append(e1.x, e1.y >> 8);
                    __builtin_amdgcn_sched_barrier(0);
                }
                held = e2.x;
                held8 = e2.y >> 8;
                const uint32_t all = two + e2.y;
                row8 += all >> 8;
                const uint32_t p = pos + (all & 63u);
                const bool cross = p >= 32u;
                pos = p & 31u;
                lo = cross ? hi : lo;
                hi = cross ? nx : hi;
                nx = cross ? pending : nx;
                next_row = cross ? min(next_row + 1u, pad_row) : next_row;
            } while (static_cast<int32_t>(row8) < target8);
            column.append(held, held8);
            column.flush();
        }
        if (lane.wave_start < first + kTileSteps) {
            // Rows at and past a stream's overflow start, from its tail.
            const uint8_t *const tail = lane.lds ? nullptr : lane.tail;
            for (int r = max(lane.start - first, 0); r < kTileSteps; ++r) {
                const int32_t i = lane.offset + (first + r - lane.start);
                const uint32_t byte = tail != nullptr ? tail[i] : tail_lds[i];
                column.base[(r >> 2) * kQuadBytes + (r & 3)] = static_cast<uint8_t>(byte + 127u);
            }
        }
        GroupSides next;
        fetch_group_sides(next, side_rsrc, first + kTileSteps, S);
        __builtin_amdgcn_wave_barrier();
        store_tile(tile, sides, out_rsrc, first, row_base, full, valid);
        __builtin_amdgcn_wave_barrier();
        sides = next;
        // Rows past the tile's end move to its start.
        uint32_t moved[kTileSpare / 4];
#pragma unroll
        for (int k = 0; k < kTileSpare / 4; ++k)
            moved[k] = *reinterpret_cast<const TileDword *>(
                column.base + (kTileSteps / 4 + k) * kQuadBytes);
#pragma unroll
        for (int k = 0; k < kTileSpare / 4; ++k)
            *reinterpret_cast<TileDword *>(column.base + k * kQuadBytes) = moved[k];
        column.row8 -= 8 * kTileSteps;
    }
}

__global__ __launch_bounds__(kLanes) void decode_kernel_grouped(
    const int32_t *__restrict__ encoded, const uint8_t *__restrict__ side,
    uint16_t *__restrict__ output, const int32_t *__restrict__ shifted_decode,
    const int32_t *__restrict__ center_ptr, int64_t n_blocks, int64_t logical_numel, int S,
    int W, int rare, lct_overflow ov, int has_overlay) {
    decode_block_grouped(encoded, side, output, shifted_decode, center_ptr, n_blocks,
                         logical_numel, S, W, rare, ov, has_overlay, blockIdx.x);
}

__global__ __launch_bounds__(kLanes) void decode_batch_kernel_grouped(DecodeBatch batch) {
    const int32_t b = static_cast<int32_t>(blockIdx.x);
    const int j = batch_job(batch, b);
    const DecodeBatchJob &job = batch.jobs[j];
    decode_block_grouped(job.encoded, job.side, job.output, job.shifted_decode, job.center,
                         job.n_blocks, job.logical_numel, job.steps, job.fixed_words, job.rare,
                         job.ov, job.has_overlay, b - batch.first_block[j]);
}

// The current device's CUs and the workgroups of each decoder that it holds at
// once for W payload words (CUs x workgroups per CU at that kernel's LDS),
// looked up once per device and W.
struct DecoderSlots {
    int32_t cus, wide, compact, grouped;
};

constexpr int kSlotDevices = 64;
constexpr size_t kLdsGrant = 1280;
std::atomic<uint64_t> g_decoder_slots[kSlotDevices][kMaxWords + 1];   // CUs << 24 | 8 bits each

// lct_set_decoder's choice (LCT_DECODER_*).
std::atomic<int32_t> g_decoder_mode{LCT_DECODER_AUTO};

int32_t decoder_slots(int W, DecoderSlots *slots) {
    int device = 0;
    if (hipError_t e = hipGetDevice(&device)) return static_cast<int32_t>(e);
    if (device < 0 || device >= kSlotDevices || W < 0 || W > kMaxWords) return LCT_E_ARG;
    uint64_t cached = g_decoder_slots[device][W].load(std::memory_order_relaxed);
    if (cached == 0) {
        int cus = 0;
        if (hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount,
                                                 device))
            return static_cast<int32_t>(e);
        const size_t lds = static_cast<size_t>(register_stage_bytes(W));
        const void *kernels[3] = {reinterpret_cast<const void *>(decode_kernel),
                                  reinterpret_cast<const void *>(decode_kernel_compact),
                                  reinterpret_cast<const void *>(decode_kernel_grouped)};
        for (int k = 0; k < 3; ++k) {
            // LDS is granted in units of kLdsGrant, which the lookup leaves out
            // (compact at W = 22: 23056 bytes, 6 workgroups per CU and not 7:
            // 32.4 us at 1536 blocks, 41.3 at 1600).
            hipFuncAttributes attributes;
            if (hipError_t e = hipFuncGetAttributes(&attributes, kernels[k]))
                return static_cast<int32_t>(e);
            const size_t fixed = attributes.sharedSizeBytes;
            const size_t granted = (fixed + lds + kLdsGrant - 1) / kLdsGrant * kLdsGrant;
            int per_cu = 0;
            if (hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
                    &per_cu, kernels[k], kLanes, granted - fixed))
                return static_cast<int32_t>(e);
            cached |= static_cast<uint64_t>(per_cu) << (8 * k);
        }
        cached |= static_cast<uint64_t>(cus) << 24;
        g_decoder_slots[device][W].store(cached, std::memory_order_relaxed);
    }
    const int32_t cus = static_cast<int32_t>(cached >> 24);
    *slots = {cus, cus * static_cast<int32_t>(cached & 255u),
              cus * static_cast<int32_t>((cached >> 8) & 255u),
              cus * static_cast<int32_t>((cached >> 16) & 255u)};
    return LCT_OK;
}

// The decoder for a grid of n_blocks workgroups (LCT_DECODER_AUTO).  A grid that
// the grouped kernel holds at once is its own.  Just past that the others still
// run one round where it needs two, of which the second is far from full, and
// from some size on its shorter lookup chain is worth more than their fuller
// rounds.  Public decompress, us, wide / compact / grouped, last block whole |
// partial (which costs the wide and compact kernels up to 7 us for a lone block
// and next to nothing in a grid of several workgroups per CU); 256 CUs:
//   W = 12 (2048 / 2048 / 1024 held), S = 128
//      36: 15.4 / 15.7 / 12.3 | 17.6 / 17.8 / 12.3    1100: 24.6 / 25.0 / 29.7 | 25.6 / 26.7 / 29.8
//    1350: 28.8 / 28.2 / 34.0 | 29.8 / 29.0 / 34.0    2048: 42.5 / 40.3 / 45.2 | 42.2 / 40.5 / 45.1
//    2100: 45.9 / 46.6 / 44.1 | 47.2 / 47.7 / 44.1    2400: 49.8 / 51.6 / 51.4 | 50.0 / 51.8 / 51.3
//    3072: 65.1 / 66.0 / 64.7 | 65.5 / 66.5 / 64.9    4096: 89.4 / 89.7 / 86.2 | 89.8 / 90.0 / 86.3
//   W = 19 (1536 / 2048 / 768), S = 128
//     800: 21.4 / 22.2 / 26.6 | 22.9 / 23.9 / 26.6    1300: 31.1 / 32.0 / 32.7 | 31.9 / 32.9 / 32.9
//    1536: 32.6 / 32.1 / 37.5 | 33.2 / 32.5 / 37.7    2048: 51.7 / 44.5 / 50.6 | 51.1 / 44.9 / 50.7
//    2560: 54.5 / 57.0 / 56.5 | 55.3 / 57.0 / 56.7    4096: 93.8 / 96.5 / 92.3 | 93.8 / 95.7 / 92.9
//   W = 22 (1280 / 1536 / 768), S = 128
//     900: 22.3 / 22.7 / 27.4 | 23.4 / 24.3 / 27.3    1450: 37.3 / 32.2 / 37.3 | 39.5 / 33.6 / 37.3
//    1600: 39.5 / 41.3 / 40.7 | 41.6 / 43.6 / 40.8    2200: 49.7 / 51.2 / 52.0 | 50.7 / 51.9 / 52.0
//    2560: 53.4 / 55.7 / 57.6 | 54.5 / 56.6 / 57.4    3328: 75.1 / 81.2 / 75.1 | 76.2 / 81.8 / 75.0
//   W = 20 (1280 / 1792 / 768), S = 256
//     900: 38.6 / 41.6 / 45.3 | 41.9 / 42.0 / 45.3    1100: 48.2 / 47.2 / 51.8 | 49.5 / 47.9 / 51.7
//    1300: 65.2 / 67.3 / 58.9 | 70.8 / 68.2 / 59.6    1536: 76.9 / 76.1 / 69.3 | 78.3 / 76.2 / 68.9
//   W = 25 (1024 / 1536 / 768), S = 256
//      36: 24.4 / 28.7 / 15.6 | 32.5 / 32.7 / 15.6     900: 38.2 / 41.6 / 43.0 | 41.3 / 42.0 / 43.1
//    1100: 56.0 / 47.8 / 51.1 | 62.6 / 49.0 / 50.6    1300: 59.9 / 66.6 / 56.1 | 65.7 / 67.9 / 57.4
//    1536: 70.2 / 74.8 / 66.5 | 74.2 / 74.6 / 66.5    4096: 180 / 191 / 171 | 186 / 191 / 171
// At S = 256 every kernel slows down where its output comes near 160 MiB (5
// blocks per CU), the compact one most and from 4.7 blocks per CU on in some
// runs (W = 20, 1215 blocks: 49 / 47 / 51 or 58 / 65 / 54): the line lies below.
// A batched launch, which has no compact form, takes 48.8 | 52.0 wide and
// 51.5 | 51.6 grouped at 1100 blocks of W = 20, and 50.3 | 64.1 and 50.5 | 57.9
// at 1200.
enum class Decoder { kWide, kCompact, kGrouped };

constexpr Decoder choose_decoder(int64_t n_blocks, int S, const DecoderSlots &slots) {
    const int64_t n = n_blocks, cus = slots.cus;
    if (n <= slots.grouped) return Decoder::kGrouped;
    if (S == 256) {
        if (2 * n > 9 * cus) return Decoder::kGrouped;
        if (n > 4 * cus && n <= slots.compact) return Decoder::kCompact;
        return n <= slots.wide ? Decoder::kWide : Decoder::kGrouped;
    }
    // The compact kernel where only it holds the grid, and from 5.5 blocks per CU.
    if (n <= slots.compact && (n > slots.wide || 2 * n >= 11 * cus)) return Decoder::kCompact;
    if (n <= slots.wide) return Decoder::kWide;
    // None holds it: the wide kernel's larger rounds where the grouped one has
    // three workgroups per CU.
    return slots.grouped < 4 * cus && n <= 12 * cus ? Decoder::kWide : Decoder::kGrouped;
}

// The table's grids.
constexpr bool chooses(const DecoderSlots &slots, int S, int64_t n, Decoder decoder) {
    return choose_decoder(n, S, slots) == decoder;
}
constexpr DecoderSlots kW12{256, 2048, 2048, 1024}, kW19{256, 1536, 2048, 768},
    kW22{256, 1280, 1536, 768}, kW20{256, 1280, 1792, 768}, kW25{256, 1024, 1536, 768};
static_assert(chooses(kW12, 128, 36, Decoder::kGrouped) && chooses(kW12, 128, 1100, Decoder::kWide)
              && chooses(kW12, 128, 2048, Decoder::kCompact)
              && chooses(kW12, 128, 2100, Decoder::kGrouped)
              && chooses(kW12, 128, 4096, Decoder::kGrouped));
static_assert(chooses(kW19, 128, 800, Decoder::kWide) && chooses(kW19, 128, 1300, Decoder::kWide)
              && chooses(kW19, 128, 1536, Decoder::kCompact)
              && chooses(kW19, 128, 2048, Decoder::kCompact)
              && chooses(kW19, 128, 2560, Decoder::kWide)
              && chooses(kW19, 128, 4096, Decoder::kGrouped));
static_assert(chooses(kW22, 128, 900, Decoder::kWide) && chooses(kW22, 128, 1450, Decoder::kCompact)
              && chooses(kW22, 128, 1600, Decoder::kWide)
              && chooses(kW22, 128, 3328, Decoder::kGrouped));
static_assert(chooses(kW20, 256, 900, Decoder::kWide) && chooses(kW20, 256, 1100, Decoder::kCompact)
              && chooses(kW20, 256, 1300, Decoder::kGrouped));
static_assert(chooses(kW25, 256, 36, Decoder::kGrouped) && chooses(kW25, 256, 900, Decoder::kWide)
              && chooses(kW25, 256, 1100, Decoder::kCompact)
              && chooses(kW25, 256, 1536, Decoder::kGrouped));

}  // namespace
}  // namespace lct

using namespace lct;

extern "C" int32_t lct_decode(const int32_t *encoded, const uint8_t *side, int16_t *output,
                              const int32_t *shifted_decode, const int32_t *center,
                              int64_t size, int64_t logical_numel, lct_geometry g,
                              int32_t rare_length, const lct_overflow *overflow,
                              hipStream_t stream) {
    if (!encoded || !side || !output || !shifted_decode || !center) return LCT_E_NULL;
    if (!geometry_ok(g)) return LCT_E_GEOMETRY;
    if (logical_numel <= 0 || size <= 0 || size % g.block_symbols != 0
        || logical_numel > size || logical_numel <= size - g.block_symbols)
        return LCT_E_SIZE;
    if (rare_length < 0 || rare_length > 8) return LCT_E_ARG;
    if ((reinterpret_cast<uintptr_t>(encoded) & 15) != 0) return LCT_E_ARG;
    lct_overflow ov{};
    if (overflow != nullptr) {
        if (!overflow->lanes || !overflow->starts || !overflow->tail || !overflow->blocks)
            return LCT_E_NULL;
        if (overflow->descriptor != nullptr && overflow->count == nullptr) return LCT_E_NULL;
        ov = *overflow;
    }
    const int64_t n_blocks = size / g.block_symbols;
    if (n_blocks > 0x7FFFFFFF) return LCT_E_SIZE;
    // Rows 0..2 of every stream start in registers (W = 2 or 3 never occurs in
    // a reference geometry).
    if (g.fixed_words <= kRegisterRows) return LCT_E_GEOMETRY;
    const size_t lds = static_cast<size_t>(register_stage_bytes(g.fixed_words));
    DecoderSlots slots;
    if (int32_t e = decoder_slots(g.fixed_words, &slots)) return e;
    Decoder decoder = choose_decoder(n_blocks, g.steps, slots);
    switch (g_decoder_mode.load(std::memory_order_relaxed)) {
    case LCT_DECODER_WIDE: decoder = Decoder::kWide; break;
    case LCT_DECODER_COMPACT: decoder = Decoder::kCompact; break;
    case LCT_DECODER_GROUPED: decoder = Decoder::kGrouped; break;
    default: break;
    }
    const auto kernel = decoder == Decoder::kGrouped   ? decode_kernel_grouped
                        : decoder == Decoder::kCompact ? decode_kernel_compact
                                                       : decode_kernel;
    if (hipError_t e = reserve_dynamic_lds(reinterpret_cast<const void *>(kernel), lds))
        return static_cast<int32_t>(e);
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(n_blocks)), dim3(kLanes), lds,
                       stream, encoded, side, reinterpret_cast<uint16_t *>(output),
                       shifted_decode, center, n_blocks, logical_numel, g.steps, g.fixed_words,
                       rare_length, ov, overflow != nullptr ? 1 : 0);
    return static_cast<int32_t>(hipGetLastError());
}

extern "C" int32_t lct_set_decoder(int32_t mode) {
    if (mode != LCT_DECODER_AUTO && mode != LCT_DECODER_WIDE && mode != LCT_DECODER_COMPACT
        && mode != LCT_DECODER_GROUPED)
        return LCT_E_ARG;
    g_decoder_mode.store(mode, std::memory_order_relaxed);
    return LCT_OK;
}

extern "C" int32_t lct_decode_batch(const lct_decode_job *jobs, int32_t n_jobs,
                                    hipStream_t stream) {
    if (!jobs) return LCT_E_NULL;
    if (n_jobs <= 0 || n_jobs > LCT_MAX_DECODE_BATCH) return LCT_E_ARG;
    DecodeBatch batch{};
    batch.n_jobs = n_jobs;
    int64_t total = 0;
    int32_t max_words = 0;
    int32_t max_steps = 0;
    for (int32_t j = 0; j < n_jobs; ++j) {
        const lct_decode_job &in = jobs[j];
        if (!in.encoded || !in.side || !in.output || !in.shifted_decode || !in.center)
            return LCT_E_NULL;
        const lct_geometry &g = in.geometry;
        if (!geometry_ok(g)) return LCT_E_GEOMETRY;
        if (in.logical_numel <= 0 || in.size <= 0 || in.size % g.block_symbols != 0
            || in.logical_numel > in.size || in.logical_numel <= in.size - g.block_symbols)
            return LCT_E_SIZE;
        if (in.rare_length < 0 || in.rare_length > 8) return LCT_E_ARG;
        if ((reinterpret_cast<uintptr_t>(in.encoded) & 15) != 0) return LCT_E_ARG;
        if (g.fixed_words <= kRegisterRows) return LCT_E_GEOMETRY;
        if (in.has_overflow) {
            const lct_overflow &o = in.overflow;
            if (!o.lanes || !o.starts || !o.tail || !o.blocks) return LCT_E_NULL;
            if (o.descriptor != nullptr && o.count == nullptr) return LCT_E_NULL;
        }
        const int64_t n_blocks = in.size / g.block_symbols;
        batch.first_block[j] = static_cast<int32_t>(total);
        total += n_blocks;
        if (total > 0x7FFFFFFF) return LCT_E_SIZE;
        DecodeBatchJob &out = batch.jobs[j];
        out.encoded = in.encoded;
        out.side = in.side;
        out.output = reinterpret_cast<uint16_t *>(in.output);
        out.shifted_decode = in.shifted_decode;
        out.center = in.center;
        out.n_blocks = n_blocks;
        out.logical_numel = in.logical_numel;
        out.steps = g.steps;
        out.fixed_words = g.fixed_words;
        out.rare = in.rare_length;
        out.has_overlay = in.has_overflow ? 1 : 0;
        out.ov = in.has_overflow ? in.overflow : lct_overflow{};
        max_steps = g.steps > max_steps ? g.steps : max_steps;
        max_words = g.fixed_words > max_words ? g.fixed_words : max_words;
    }
    batch.first_block[n_jobs] = static_cast<int32_t>(total);
    const size_t lds = static_cast<size_t>(register_stage_bytes(max_words));
    DecoderSlots slots;
    if (int32_t e = decoder_slots(max_words, &slots)) return e;
    slots.compact = 0;   // no batched form
    const int32_t mode = g_decoder_mode.load(std::memory_order_relaxed);
    const bool wide = mode == LCT_DECODER_WIDE
                      || (mode != LCT_DECODER_GROUPED
                          && choose_decoder(total, max_steps, slots) == Decoder::kWide);
    const auto kernel = wide ? decode_batch_kernel : decode_batch_kernel_grouped;
    if (hipError_t e = reserve_dynamic_lds(reinterpret_cast<const void *>(kernel), lds))
        return static_cast<int32_t>(e);
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(total)), dim3(kLanes), lds, stream,
                       batch);
    return static_cast<int32_t>(hipGetLastError());
}
