// Single-pass pointwise update with compressed output (gfx950).
//
// The reference's compressed-output path (LCT/codec/pointwise.py:262-278)
// runs the fused pointwise kernel with COMPRESSED_OUTPUT, which writes the
// result's side bytes and exponent bytes to HBM
// (LCT/kernels/generic/pointwise.py:43-65), and then re-encodes them through
// encode_components(precomputed=True) (LCT/codec/encode.py:22-186): a center
// estimated from up to 4096 sampled exponent bytes of the result
// (LCT/kernels/common/tables.py:9-49), the encoder kernel
// (LCT/kernels/generic/encode.py:10-169), the block scan and the compaction.
// The result's exponent and side bytes make a round trip through HBM between
// the two passes.  Here they never leave the chip:
//
//  * pointwise_sample_kernel computes the operation's result only at the
//    sampled positions, decoding each sampled stream's prefix from its payload
//    words, and writes the exponent sum and count of each group of 64 samples;
//  * pointwise_encode_kernel reduces those sums to the result's center in
//    every workgroup, shifts the result distribution's encode table by it, and
//    then, per codec block, decodes A, applies the operation with the dense
//    operand B and encodes the result in the same pass.  Its outputs are the
//    encoder's: side bytes, every payload word, extra starts and the block
//    summaries.  Rows that an overflowing stream cannot hold also get the
//    result's exponent bytes written (logical order, those rows only), which
//    is where the compaction reads their tails, as in the precomputed path.
//
// Both directions work in quads of symbols (update_core.h).  The encoder side
// writes each payload word straight to HBM when the word completes (one 4-byte
// store by the lanes whose word a quad completed, merged in L2), so the
// workgroup's LDS holds only A's payload (30.9 KiB in all at W = 25).  The
// result's side bytes leave with the default cache policy: a wave writes 64
// bytes of each 128-byte row line, and non-temporal stores of half lines wrote
// 16% more than the side bytes (C4: 73.6 MB against 62.9 MB per launch; with
// the default policy 63.3 MB, at equal kernel time).
//
// Measured (kernel trace, three operand sets in turn; pairs of symbols, a
// register or LDS window per pair and one step loop per overlay, before ->
// quads): pointwise_encode_kernel 64.0 -> 61.1 us at 688 blocks, 38.2 -> 36.2
// at one; dual_encode_kernel 75.6 -> 69.2 and 46.7 -> 43.0.  A ragged tensor's
// last block runs the same loop (the whole momentum step at 767 blocks, ragged:
// 75.8 us, against 150 us with a separate loop for partial blocks).  With 203
// and 275 VALU instructions per 8 steps and 2.7 waves per SIMD, the VALU is 44
// and 55% busy; the rest is waits for the lookups' LDS round trips.
#include <algorithm>

#include "batch.h"
#include "reserve.h"
#include "update_core.h"

namespace lct {
namespace {

// Cache policy of the result's side-byte stores: the default (see above).
constexpr int kSideStore = 0;

struct OperandA {
    const int32_t *encoded;
    const uint8_t *side;
    const int32_t *shifted_decode;
    const int32_t *center;
    lct_overflow ov;
    int32_t has_overlay;
};

struct OpArgs {
    const float *alpha;
    const float *beta;
    int32_t op;
    int32_t alpha_is_one;
    int32_t beta_is_one;
};

// The in-launch overflow bookkeeping of the *_encode_fused launches (control
// == nullptr: the block summaries go to `summaries` for a later launch).
struct KernelBookkeeping {
    uint64_t *control;
    uint32_t epoch;
    int32_t *counts;
    int32_t *blocks;
    int32_t *descriptor;
    int32_t *buffer_meta;
    int32_t max_free_regions;
    lct_pending_frees frees;
    int32_t lock_spins;
    int32_t polls;
    // In-launch center sampling of the two-operand launch (sample_groups > 0):
    // workgroups g < sample_groups publish sample group g's partial sums in
    // control[g] (tagged), and every block reads the center from there
    // instead of from `partials`.
    const uint16_t *a_samples;
    const uint16_t *b_samples;
    uint16_t *result_samples;
    int64_t sample_size;
    int32_t sample_groups;
};

// Publish sample group `group`'s kept-exponent sum and count (one wave,
// compress.hip's layout: sum as int16 in bits 16..31, count in bits 0..15).
__device__ __forceinline__ void publish_sample_group(const KernelBookkeeping &bk, int64_t group,
                                                     int32_t sum, int32_t kept) {
    if (threadIdx.x == 0) {
        const uint32_t value = (static_cast<uint32_t>(static_cast<uint16_t>(sum)) << 16)
                               | static_cast<uint32_t>(kept);
        control_store(bk.control + group, tagged_word(bk.epoch, value));
    }
}

// Workgroup 0's share of the result's shifted decode table: the base
// table's 1024 entries, 4 per thread, loaded at the start of its prologue
// (with the other loads) and shifted once the center is known, so that the
// workgroup that also writes the table has no extra memory round trip.
struct BaseDecodeShare {
    int32_t v[1024 / kLanes];
};

__device__ __forceinline__ BaseDecodeShare load_base_decode(const int32_t *__restrict__ base_decode,
                                                            bool needed) {
    BaseDecodeShare b{};
    if (needed) {
#pragma unroll
        for (int k = 0; k < 1024 / kLanes; ++k) b.v[k] = base_decode[threadIdx.x + k * kLanes];
    }
    return b;
}

__device__ __forceinline__ void store_shifted_decode(int32_t *__restrict__ out,
                                                     const BaseDecodeShare &b, int32_t center) {
#pragma unroll
    for (int k = 0; k < 1024 / kLanes; ++k)
        out[threadIdx.x + k * kLanes] = shifted_decode_entry(b.v[k], center);
}

// After a block (every thread, past the summary's barriers): its overflow
// count and tail bytes go to `summaries`, or -- in a fused launch (kBooked:
// its own kernel instantiation, so the separate launch's kernel holds none of
// the bookkeeping's arguments in registers) -- to the control array as a
// tagged word, and workgroup 0 then does the bookkeeping
// of the one-launch compress: with a buffer the lock, the deferred frees and
// the free list in `lds_free_list` (the payload stage, free by now), the
// polled scan into the block metadata and the overflow-block list, and the
// reservation (lct_prefix_allocate / lct_allocate_compact's results).
template <bool kBooked, class Book>
__device__ __forceinline__ void publish_block(const KernelBookkeeping &bk,
                                              int32_t *__restrict__ summaries, int64_t block,
                                              int64_t n_blocks, int32_t count, int32_t bytes,
                                              int32_t *lds_free_list, int32_t *lds_words,
                                              Book book, bool failed = false) {
    if (!kBooked) {
        if (threadIdx.x == 0) {
            summaries[block] = count;
            summaries[n_blocks + block] = bytes;
        }
        return;
    }
    if (threadIdx.x == 0) {
        // count <= 256 and bytes <= 256 * 256 fit 9 and 17 bits; a block
        // whose center did not arrive is marked failed.
        const uint32_t value = failed ? (kFailedBlock << 17)
                                      : (static_cast<uint32_t>(count) << 17)
                                            | static_cast<uint32_t>(bytes);
        control_store(bk.control + kControlPartials + block, tagged_word(bk.epoch, value));
    }
    if (block != 0) return;
    PolledSummaries polled{bk.control, bk.epoch, static_cast<int32_t>(n_blocks), bk.polls, false};
    if (bk.buffer_meta != nullptr) {
        LdsReserve<false> reserve{
            AllocatorMeta(bk.buffer_meta, bk.max_free_regions, bk.lock_spins), bk.descriptor,
            bk.frees, lds_free_list, {}, -1, kStatusOk};
        book(polled, summaries, bk.counts, bk.blocks, static_cast<int32_t>(n_blocks), reserve,
             lds_words);
    } else {
        NoReserve reserve;
        scan_allocate<false>(polled, summaries, bk.counts, bk.blocks,
                             static_cast<int32_t>(n_blocks), reserve);
    }
}

// Overflow start and tail byte index of one stream (block, lane) of A, from
// the block's entry list (ascending lanes, tails concatenated in entry order:
// LCT/kernels/generic/compaction.py:137-228, decode.py:195-240).  `start` is S
// when the stream does not overflow.
__device__ __forceinline__ void stream_overlay(const lct_overflow &ov, bool present, int64_t block,
                                               int64_t n_blocks, int32_t lane, int S,
                                               int32_t &start, int64_t &tail_index) {
    start = S;
    tail_index = 0;
    if (!present) return;
    int32_t count = ov.blocks[block];
    if (ov.descriptor != nullptr && ov.descriptor[2] != 0) count = 0;
    if (count <= 0) return;
    int64_t lane_off = 0, start_off = 0, tail_base = ov.base;
    if (ov.descriptor != nullptr) {
        const int64_t arena = ov.descriptor[0];
        const int64_t total = ov.count[0];
        lane_off = arena;
        start_off = arena + total;
        tail_base = arena + 2 * total;
    }
    const int32_t first = ov.blocks[n_blocks + block];
    int64_t offset = tail_base + ov.blocks[2 * n_blocks + block];
    for (int32_t e = 0; e < count; ++e) {
        const int32_t entry_lane = ov.lanes[lane_off + first + e];
        const int32_t entry_start = ov.starts[start_off + first + e];
        if (entry_lane == lane) {
            start = entry_start;
            tail_index = offset;
            return;
        }
        offset += S - entry_start;
    }
}

// One sample per thread: the result's exponent at sample position i.  A's
// value there comes from a_samples (A's values at the same positions, recorded
// when A was made) or, without it, from A's streams: the sampled stream's W
// words are staged in this thread's LDS column and its pairs decoded up to the
// sample's step.  The result's values go to result_samples when given.
// Sample group `group` (the single launch's blockIdx.x); `words`: the dynamic
// LDS, (W + 1) rows x kSampleGroup.
__device__ __forceinline__ void pointwise_sample_group(
    const OperandA &a, const uint16_t *__restrict__ a_samples, const uint16_t *__restrict__ other,
    const OpArgs &args, int64_t n_blocks, int64_t logical_numel, int64_t sample_size, int S,
    int W, int rare, int32_t *__restrict__ partials, uint16_t *__restrict__ result_samples,
    int64_t group, uint32_t *words) {
    __shared__ DecodeTables tb;
    const int t = threadIdx.x;
    if (a_samples != nullptr) {
        const int64_t i = group * kSampleGroup + t;
        const bool active = i < sample_size;
        const int shift = __builtin_ctzll(static_cast<uint64_t>(sample_size));
        uint32_t result = 0;
        if (active) {
            const int64_t pos = sample_position(i, logical_numel, sample_size, shift);
            const OpParams p = load_op_params(args.op, args.alpha_is_one, args.beta_is_one,
                                              args.alpha, args.beta);
            result = apply_op(p, a_samples[i], other[pos]);
            if (result_samples != nullptr) result_samples[i] = static_cast<uint16_t>(result);
        }
        const int32_t exp = static_cast<int32_t>((result >> 7) & 255u) - 127;
        const bool keep = active && exp >= -120;
        const int32_t sum = wave_sum(keep ? exp : 0);
        const int32_t kept = wave_sum(keep ? 1 : 0);
        if (t == 0) {
            partials[2 * group] = sum;
            partials[2 * group + 1] = kept;
        }
        return;
    }
    int32_t packed[256 / kSampleGroup];
#pragma unroll
    for (int k = 0; k < 256 / kSampleGroup; ++k) packed[k] = a.shifted_decode[t + k * kSampleGroup];
    const int32_t center = a.center[0];
    const OpParams p = load_op_params(args.op, args.alpha_is_one, args.beta_is_one, args.alpha,
                                      args.beta);

    const int64_t i = group * kSampleGroup + t;
    const bool active = i < sample_size;
    const int shift = __builtin_ctzll(static_cast<uint64_t>(sample_size));
    const int64_t pos = active ? sample_position(i, logical_numel, sample_size, shift) : 0;
    const int64_t row = pos / kLanes;                 // storage row of the sample
    const int32_t lane = static_cast<int32_t>((pos % kLanes) ^ (row & 254));
    const int64_t block = row >> (S == 128 ? 7 : 8);   // S is 128 or 256
    const int32_t step = static_cast<int32_t>(row & (S - 1));
    const int64_t n_streams = n_blocks * kLanes;
    // The stream's words go straight to this thread's LDS column (row w at
    // words[w * 64 + t]); all W loads are in flight at once.  Inactive lanes
    // read stream 0.
    const int32_t *column = a.encoded + (active ? block * kLanes + lane : 0);
    for (int w = 0; w < W; ++w)
        __builtin_amdgcn_global_load_lds(
            column + w * n_streams,
            (__attribute__((address_space(3))) void *)(words + w * kSampleGroup), 4, 0, 0);
    words[W * kSampleGroup + t] = 0u;
    const uint32_t sm = active ? a.side[row * kLanes + lane] : 0u;
    const uint32_t b = active ? other[pos] : 0u;
#pragma unroll
    for (int k = 0; k < 256 / kSampleGroup; ++k)
        build_decode_entry(tb, t + k * kSampleGroup, packed[k], center);
    int32_t start;
    int64_t tail_index;
    stream_overlay(a.ov, active && a.has_overlay != 0, block, n_blocks, lane, S, start, tail_index);
    wait_memory();
    __syncthreads();   // decode tables and staged words

    uint32_t field = 0;
    if (step >= start) {
        field = tail_field(a.ov.tail[tail_index + (step - start)]);
    } else if (active) {
        // Steps before `start` hold payload codes; so do all earlier steps of
        // the stream, none of which is padding (their logical offsets are
        // below this sample's).
        StreamCursorT<kSampleGroup> cursor;
        cursor.init(words + t, &tb, static_cast<uint32_t>(W), rare);
        for (int pair = 0; pair < step / 2; ++pair) {
            uint32_t f0, f1;
            cursor.advance(cursor.next_fields(f0, f1));
        }
        uint32_t f0, f1;
        cursor.next_fields(f0, f1);
        field = (step & 1) ? f1 : f0;
    }
    const uint32_t result = apply_op(p, join_entry(field, sm), b);
    if (active && result_samples != nullptr) result_samples[i] = static_cast<uint16_t>(result);
    const int32_t exp = static_cast<int32_t>((result >> 7) & 255u) - 127;
    const bool keep = active && exp >= -120;
    const int32_t sum = wave_sum(keep ? exp : 0);
    const int32_t kept = wave_sum(keep ? 1 : 0);
    if (t == 0) {
        partials[2 * group] = sum;
        partials[2 * group + 1] = kept;
    }
}

__global__ __launch_bounds__(kSampleGroup) void pointwise_sample_kernel(
    OperandA a, const uint16_t *__restrict__ a_samples, const uint16_t *__restrict__ other,
    OpArgs args, int64_t n_blocks, int64_t logical_numel, int64_t sample_size, int S, int W,
    int rare, int32_t *__restrict__ partials, uint16_t *__restrict__ result_samples) {
    extern __shared__ uint32_t words[];   // (W + 1) rows x kSampleGroup
    pointwise_sample_group(a, a_samples, other, args, n_blocks, logical_numel, sample_size, S, W,
                           rare, partials, result_samples, blockIdx.x, words);
}

// ---- the fused decode -> operation -> encode kernel
//
// Memory operations are arranged for gfx9's single load/store counter
// (vmcnt): a chunk's A side bytes and B words are fetched two chunks ahead,
// before the previous chunk's stores are issued, and every store is
// unconditional -- lanes that must not write get an out-of-range buffer offset,
// which the hardware drops.  The compiler can then wait for exactly the loads
// it needs without also waiting for recent stores.
//
// Each 8-step half is emitted (arithmetic, side bytes, codes) while the next
// one is decoded; the two are independent, and scheduling barriers put a piece
// of the emitting behind each of the decode's dependent lookups.

struct UpdateIo {
    __amdgpu_buffer_rsrc_t side;       // A's side bytes (storage order)
    __amdgpu_buffer_rsrc_t other;      // B, BF16 in logical order
    __amdgpu_buffer_rsrc_t side_out;   // result side bytes (storage order)
    __amdgpu_buffer_rsrc_t exponents;  // result exponent bytes of overflow rows (logical order)
};

// B words of the 16-step chunk at `first` (one 4-byte word per lane per step
// pair, lane-pair layout), or zeros without memory traffic past the block's
// last step.  A partial block's words are read by halves: one that straddles
// the tensor's end would read as 0 whole.
template <bool kFull>
__device__ __forceinline__ void fetch_b_chunk(uint32_t (&bw)[kChunkSteps / 2],
                                              const UpdateIo &io, const LanePair &lp,
                                              int64_t row_base, int first, int S) {
    const uint32_t base = first < S
                              ? lp.offset2 ^ static_cast<uint32_t>((row_base + first) & 254) * 2u
                              : kOutOfRange;   // stays out of range under the XOR
#pragma unroll
    for (int j = 0; j < kChunkSteps; j += 2) {
        const uint32_t off = base ^ static_cast<uint32_t>(2 * j);
        const int row = (first + j) * kLanes * 2;
        if (kFull) {
            bw[j / 2] = __builtin_amdgcn_raw_buffer_load_b32(io.other, off, row, 0);
        } else {
            const uint32_t low = __builtin_amdgcn_raw_buffer_load_b16(io.other, off, row, 0);
            const uint32_t high = __builtin_amdgcn_raw_buffer_load_b16(io.other, off + 2u, row, 0);
            bw[j / 2] = low | (high << 16);
        }
    }
}

// A's side bytes and B's words of one chunk.
struct Prefetch {
    SideChunk side;
    uint32_t b[kChunkSteps / 2];
};

// What a lane walks a block with.
struct UpdateWalk {
    QuadCursor cursor;
    LaneOverlay lane;
    const uint8_t *tail_lds;
    StreamWriter writer;
    const uint2 *enc;
    uint8_t *slice;        // this wave's 16 rows of side bytes
    OpParams p;
    int64_t row_base;
    uint32_t valid;        // elements of the block inside the tensor
};

// Emit the half at `first` (f: its entries; rows: its side bytes in the slice;
// bw: its B words) while decoding the next half into f.  kFast: every code is
// known to fit.
template <bool kFull, int kForm, bool kFast>
__device__ __forceinline__ void update_half(UpdateWalk &u, uint32_t (&f)[kHalfSteps],
                                            uint8_t *rows, const uint32_t *bw, const UpdateIo &io,
                                            const LanePair &lp, int first, int S) {
    const uint32_t mask = static_cast<uint32_t>((u.row_base + first) & 254);
    Quad q;
    u.cursor.first(q);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t sa[kHalfSteps];
    float b[kHalfSteps], x[kHalfSteps];
#pragma unroll
    for (int k = 0; k < kHalfSteps; ++k) sa[k] = side_byte(rows, k);
#pragma unroll
    for (int p = 0; p < kHalfSteps / 2; ++p) pair_unpack16(lp, bw[p], b[2 * p], b[2 * p + 1]);
    __builtin_amdgcn_sched_barrier(0);
    u.cursor.second(q);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kHalfSteps; ++k)
        x[k] = apply_form<kForm>(u.p, __uint_as_float(join_float(f[k], sa[k])), b[k]);
    __builtin_amdgcn_sched_barrier(0);
    u.cursor.third(q);
    __builtin_amdgcn_sched_barrier(0);
    HalfEmit h;
    round_half<kFull>(h, x, first, mask, u.valid);
    store_half_sides(h, rows);
    __builtin_amdgcn_sched_barrier(0);
    u.cursor.fourth(q);
    __builtin_amdgcn_sched_barrier(0);
    look_up_quad<kFull>(h, u.enc, 0, first, mask, u.valid);
    __builtin_amdgcn_sched_barrier(0);
    u.cursor.finish(q, f);
    u.cursor.first(q);
    __builtin_amdgcn_sched_barrier(0);
    look_up_quad<kFull>(h, u.enc, 1, first, mask, u.valid);
    __builtin_amdgcn_sched_barrier(0);
    u.cursor.second(q);
    __builtin_amdgcn_sched_barrier(0);
    if (kFast) {
        const QuadCodes c0(h, 0), c1(h, 1);
        __builtin_amdgcn_sched_barrier(0);
        u.cursor.third(q);
        __builtin_amdgcn_sched_barrier(0);
        put_half(c0, c1, u.writer);
    } else {
        u.cursor.third(q);
        put_half_by_pairs(h, u.writer, first, mask, io.exponents);
    }
    __builtin_amdgcn_sched_barrier(0);
    u.cursor.fourth(q);
    u.cursor.finish(q, f + 4);
    overlay_half(u.lane, u.tail_lds, first + kHalfSteps, S, f);
}

// The 16-step chunk at c, whose side bytes and B words pf holds; refills pf
// with chunk c + 32's.
template <bool kFull, int kForm>
__device__ __forceinline__ void update_chunk(UpdateWalk &u, uint32_t (&f)[kHalfSteps],
                                             Prefetch &pf, const UpdateIo &io, const LanePair &lp,
                                             int c, int S) {
    const uint32_t voffset = side_fetch_offset();
    store_side_chunk(u.slice, pf.side);
    uint32_t bw[kChunkSteps / 2];
#pragma unroll
    for (int k = 0; k < kChunkSteps / 2; ++k) bw[k] = pf.b[k];
    const int ahead = c + 2 * kChunkSteps;
    pf.side = fetch_side_chunk(io.side, ahead < S ? voffset : kOutOfRange, ahead);
    fetch_b_chunk<kFull>(pf.b, io, lp, u.row_base, ahead, S);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        uint8_t *const rows = u.slice + half * kHalfSteps * kWave;
        const uint32_t *const b = bw + half * kHalfSteps / 2;
        const int first = c + half * kHalfSteps;
        if (__builtin_expect(u.writer.fits_half(), 1))
            update_half<kFull, kForm, true>(u, f, rows, b, io, lp, first, S);
        else
            update_half<kFull, kForm, false>(u, f, rows, b, io, lp, first, S);
    }
    // The slice now holds the chunk's result side bytes.
    const uint4 q = reinterpret_cast<const uint4 *>(u.slice)[threadIdx.x & (kWave - 1)];
    store_b128<kSideStore>(q, io.side_out, voffset + static_cast<uint32_t>(c) * kLanes);
}

// A whole block.  Two copies of the prefetched data alternate, so a chunk's
// loads are issued two chunks before use and no register copy of an in-flight
// load (which would wait for it) is made.  The last half decodes eight symbols
// past the block's end, which nothing uses.
template <bool kFull, int kForm>
__device__ __forceinline__ void update_rows(UpdateWalk &u, const SideChunk &first_side,
                                            const UpdateIo &io, int S) {
    const LanePair lp;
    Prefetch even, odd;
    even.side = first_side;
    odd.side = fetch_side_chunk(io.side, side_fetch_offset(), kChunkSteps);
    fetch_b_chunk<kFull>(even.b, io, lp, u.row_base, 0, S);
    fetch_b_chunk<kFull>(odd.b, io, lp, u.row_base, kChunkSteps, S);
    uint32_t f[kHalfSteps];
    u.cursor.quad(f);
    u.cursor.quad(f + 4);
    overlay_half(u.lane, u.tail_lds, 0, S, f);
#pragma unroll 1
    for (int c = 0; c < S; c += 2 * kChunkSteps) {
        update_chunk<kFull, kForm>(u, f, even, io, lp, c, S);
        update_chunk<kFull, kForm>(u, f, odd, io, lp, c + kChunkSteps, S);
    }
}

// Codec block `block` of one fused update (the single launch's blockIdx.x);
// `stage`: the dynamic LDS, register_stage_bytes(W) (rows 3..W-1 of A's payload).
template <bool kBooked, class Book>
__device__ __forceinline__ void pointwise_encode_block(
    const OperandA &a, const uint16_t *__restrict__ other, const OpArgs &args,
    const int32_t *__restrict__ partials, int32_t n_groups,
    const int32_t *__restrict__ base_encode, const int32_t *__restrict__ base_decode,
    int32_t *__restrict__ center_out, int32_t *__restrict__ shifted_decode_out,
    uint8_t *__restrict__ side_out, int32_t *__restrict__ encoded_out,
    uint8_t *__restrict__ extra_starts, int32_t *__restrict__ summaries,
    uint8_t *__restrict__ exponents, int64_t n_blocks, int64_t logical_numel, int S, int W,
    int rare, const KernelBookkeeping &bk, int64_t block, uint32_t *stage, Book book) {
    __shared__ QuadTables tb;
    __shared__ uint2 enc[256];
    __shared__ int32_t scratch[kWavesPerBlock];
    __shared__ int32_t shared_center;
    __shared__ uint8_t tail_lds[kTailLds];
    // The overflow maps (2 KiB) and the raw encode table (1 KiB) are only used
    // before the first side chunk is stored, so they share the side slices.
    __shared__ __attribute__((aligned(16))) uint8_t side_slices[kWavesPerBlock][kChunkSteps * kWave];
    int32_t *map_start = reinterpret_cast<int32_t *>(&side_slices[0][0]);
    int32_t *map_offset = map_start + kLanes;
    int32_t *raw_encode = map_offset + kLanes;
    const int t = threadIdx.x;
    const int64_t row_base = block * S;
    const int64_t logical_base = row_base * kLanes;
    const uint32_t block_elems = static_cast<uint32_t>(S) * kLanes;
    const int64_t remaining = logical_numel - logical_base;
    const uint32_t valid = remaining < block_elems ? static_cast<uint32_t>(remaining) : block_elems;
    UpdateIo io;
    io.side = make_rsrc(a.side + logical_base, block_elems);
    io.other = make_rsrc(other + logical_base, 2u * valid);
    io.side_out = make_rsrc(side_out + logical_base, block_elems);
    io.exponents = make_rsrc(exponents + logical_base, valid);
    const SideChunk first = fetch_side_chunk(io.side, side_fetch_offset(), 0);

    // The result's center from the sampler's partial sums.
    raw_encode[t] = base_encode[t];
    center_from_partials(partials, n_groups, &shared_center);
    build_quad_tables(tb, a.shifted_decode, rare);
    const int32_t a_center = a.center[0];
    uint32_t words[kRegisterRows];
    load_register_rows(a.encoded, n_blocks * kLanes, block, words);
    stage_payload_rows(stage, a.encoded, n_blocks * kLanes, block, kRegisterRows, W);
    __syncthreads();   // center and raw encode table
    const int32_t center = shared_center;
    enc[t] = repack_encode_entry(static_cast<uint32_t>(raw_encode[byte_to_index(t, center)]));
    if (block == 0) {
        if (t == 0) center_out[0] = center;
        for (int i = t; i < 1024; i += kLanes)
            shifted_decode_out[i] = shifted_decode_entry(base_decode[i], center);
    }
    __syncthreads();   // raw_encode is no longer read (it shares the maps' LDS)
    const LaneOverlay lane = build_overlay(a.ov, a.has_overlay != 0, block, n_blocks, S, map_start,
                                           map_offset, scratch, tail_lds, kTailLds);
    // (Issued here rather than with the prologue's first loads: hoisted, the
    // measured kernel was 0.8 us slower.)
    const OpParams p = load_op_params(args.op, args.alpha_is_one, args.beta_is_one, args.alpha,
                                      args.beta);
    wait_memory();
    __syncthreads();   // payload, tails and encode table visible; maps no longer read

    UpdateWalk u;
    u.cursor.init(stage + t, &tb, static_cast<uint32_t>(W), rare, words, a_center);
    u.lane = lane;
    u.tail_lds = tail_lds;
    const uint32_t row_bytes = static_cast<uint32_t>(n_blocks * kLanes * 4);
    u.writer = StreamWriter{make_rsrc(encoded_out + block * kLanes,
                                      static_cast<uint32_t>(W - 1) * row_bytes + kLanes * 4),
                            row_bytes, static_cast<uint32_t>(t) * 4u,
                            static_cast<uint32_t>(W) * row_bytes + static_cast<uint32_t>(t) * 4u,
                            static_cast<uint32_t>(W) * 32u, 0u, 0u, 0u};
    u.writer.keep_row_bytes_in_vgpr();
    u.enc = enc;
    u.slice = side_slices[t / kWave];
    u.p = p;
    u.row_base = row_base;
    u.valid = valid;
    const bool full = valid == block_elems;
#define LCT_ROWS(FORM)                              \
    do {                                            \
        if (full) update_rows<true, FORM>(u, first, io, S);  \
        else update_rows<false, FORM>(u, first, io, S);      \
    } while (0)
    switch (form_of(args.op, args.alpha_is_one, args.beta_is_one)) {
    case kFormAxpy: LCT_ROWS(kFormAxpy); break;
    case kFormAxpby: LCT_ROWS(kFormAxpby); break;
    case kFormBxpa: LCT_ROWS(kFormBxpa); break;
    default: LCT_ROWS(kFormMul); break;
    }
#undef LCT_ROWS
    u.writer.finish();
    const bool overflow = u.writer.overflowed();
    const int32_t extra = u.writer.extra_start();
    extra_starts[block * kLanes + t] = static_cast<uint8_t>(overflow ? extra : 255);
    // Streams from bit 20 (at most 256), tail bytes in bits 0..19 (at most
    // 256 x 256): one block scan.
    const int32_t both = block_sum(overflow ? (S - extra) | (1 << 20) : 0, scratch);
    publish_block<kBooked>(bk, summaries, block, n_blocks, both >> 20, both & 0xFFFFF,
                           reinterpret_cast<int32_t *>(stage), map_start, book);
}

template <bool kBooked>
__global__ __launch_bounds__(kLanes) void pointwise_encode_kernel(
    OperandA a, const uint16_t *__restrict__ other, OpArgs args,
    const int32_t *__restrict__ partials, int32_t n_groups,
    const int32_t *__restrict__ base_encode, const int32_t *__restrict__ base_decode,
    int32_t *__restrict__ center_out, int32_t *__restrict__ shifted_decode_out,
    uint8_t *__restrict__ side_out, int32_t *__restrict__ encoded_out,
    uint8_t *__restrict__ extra_starts, int32_t *__restrict__ summaries,
    uint8_t *__restrict__ exponents, int64_t n_blocks, int64_t logical_numel, int S, int W,
    int rare, KernelBookkeeping bk) {
    extern __shared__ uint32_t stage[];   // register_stage_bytes(W)
    pointwise_encode_block<kBooked>(a, other, args, partials, n_groups, base_encode, base_decode,
                                    center_out, shifted_decode_out, side_out, encoded_out,
                                    extra_starts, summaries, exponents, n_blocks, logical_numel,
                                    S, W, rare, bk, blockIdx.x, stage, SingleBook{});
}

// ---- several fused updates of one operation in three launches
//
// A layer's weights are a few codec blocks each, so one update's sampler,
// encoder and compaction are each bound by one block's latency; the batched
// form runs up to LCT_MAX_UPDATE_BATCH tensors' samplers in one launch, their
// encoders (with the in-launch bookkeeping, buffered) in a second and their
// compactions in a third.  Workgroup w of a launch works for the last job
// whose first workgroup is at most w.  The job tables travel in the kernel
// arguments.

struct UpdateSampleJob {
    OperandA a;
    const uint16_t *a_samples;
    const uint16_t *other;
    int32_t *partials;
    uint16_t *result_samples;
    int64_t n_blocks;
    int64_t logical_numel;
    int64_t sample_size;
    int32_t steps;
    int32_t fixed_words;
    int32_t rare;
};

struct UpdateSampleBatch {
    int32_t n_jobs;
    int32_t first_group[LCT_MAX_UPDATE_BATCH + 1];
    UpdateSampleJob jobs[LCT_MAX_UPDATE_BATCH];
    OpArgs args;
};

__global__ __launch_bounds__(kSampleGroup) void pointwise_sample_batch_kernel(
    UpdateSampleBatch batch) {
    extern __shared__ uint32_t words[];   // (max W + 1) rows x kSampleGroup
    const int32_t w = static_cast<int32_t>(blockIdx.x);
    int j = 0;
    for (int k = 1; k < batch.n_jobs; ++k)
        if (w >= batch.first_group[k]) j = k;
    const UpdateSampleJob &job = batch.jobs[j];
    pointwise_sample_group(job.a, job.a_samples, job.other, batch.args, job.n_blocks,
                           job.logical_numel, job.sample_size, job.steps, job.fixed_words,
                           job.rare, job.partials, job.result_samples,
                           w - batch.first_group[j], words);
}

struct UpdateEncodeJob {
    OperandA a;
    const uint16_t *other;
    const int32_t *partials;
    const int32_t *base_encode;
    const int32_t *base_decode;
    int32_t *center_out;
    int32_t *shifted_decode_out;
    uint8_t *side_out;
    int32_t *encoded_out;
    uint8_t *extra_starts;
    int32_t *summaries;
    uint8_t *exponents;
    uint64_t *control;
    int32_t *counts;
    int32_t *blocks;
    int32_t *descriptor;
    int64_t n_blocks;
    int64_t logical_numel;
    int32_t n_groups;
    int32_t steps;
    int32_t fixed_words;
    int32_t rare;
};

struct UpdateEncodeBatch {
    int32_t n_jobs;
    int32_t first_block[LCT_MAX_UPDATE_BATCH + 1];
    UpdateEncodeJob jobs[LCT_MAX_UPDATE_BATCH];
    OpArgs args;
    int32_t *buffer_meta;
    int32_t max_free_regions;
    lct_pending_frees frees;
    uint32_t epoch;
    int32_t lock_spins;
    int32_t polls;
};

__global__ __launch_bounds__(kLanes) void pointwise_encode_batch_kernel(UpdateEncodeBatch batch) {
    extern __shared__ uint32_t stage[];   // register_stage_bytes(max W), or the free list
    const int32_t w = static_cast<int32_t>(blockIdx.x);
    int j = 0;
    for (int k = 1; k < batch.n_jobs; ++k)
        if (w >= batch.first_block[k]) j = k;
    const UpdateEncodeJob &job = batch.jobs[j];
    KernelBookkeeping bk{job.control, batch.epoch, job.counts, job.blocks, job.descriptor,
                         batch.buffer_meta, batch.max_free_regions, batch.frees,
                         batch.lock_spins, batch.polls};
    pointwise_encode_block<true>(job.a, job.other, batch.args, job.partials, job.n_groups,
                                 job.base_encode, job.base_decode, job.center_out,
                                 job.shifted_decode_out, job.side_out, job.encoded_out,
                                 job.extra_starts, job.summaries, job.exponents, job.n_blocks,
                                 job.logical_numel, job.steps, job.fixed_words, job.rare, bk,
                                 w - batch.first_block[j], stage,
                                 TableBook<UpdateEncodeBatch>{batch, j});
}

// ---- the two-compressed form: alpha * A + B with compressed output
//
// The reference's weight update (LCT/LCTensor.py:91-99 -> codec/pointwise.py:
// 159-210 with dense_output=False) runs the dual kernel with
// COMPRESSED_OUTPUT (LCT/kernels/generic/pointwise_scalar_dual.py:17-346) and
// re-encodes its components.  As for one compressed operand, the sampler
// computes the result at the sample positions and the encode kernel decodes
// both operands, applies fma(a, alpha, b) (pointwise_scalar_dual.py:226) and
// encodes the result in one pass.

// One compressed operand of the sampler whose value at the sample has to be
// decoded from its stream: the state between issuing its loads and walking.
struct SampleWalk {
    int32_t start;        // first overflow step of the sampled stream, S if none
    int64_t tail_index;   // its tail's first byte
    uint32_t sm;          // side byte at the sample
};

// Stage the sampled stream's W words into this thread's LDS column of
// `words`, read the side byte and the stream's overflow entry.
__device__ __forceinline__ void sample_issue(const OperandA &x, bool active, int64_t row,
                                             int32_t lane, int64_t block, int64_t n_blocks,
                                             int S, int W, uint32_t *words, SampleWalk &w) {
    const int t = threadIdx.x;
    const int64_t n_streams = n_blocks * kLanes;
    const int32_t *column = x.encoded + (active ? block * kLanes + lane : 0);
    for (int r = 0; r < W; ++r)
        __builtin_amdgcn_global_load_lds(
            column + r * n_streams,
            (__attribute__((address_space(3))) void *)(words + r * kSampleGroup), 4, 0, 0);
    words[W * kSampleGroup + t] = 0u;
    w.sm = active ? x.side[row * kLanes + lane] : 0u;
    stream_overlay(x.ov, active && x.has_overlay != 0, block, n_blocks, lane, S, w.start,
                   w.tail_index);
}

// The operand's BF16 bits at the sample (after the staged words and tables
// are visible): the tail byte at or after the stream's overflow start, else
// the decoded prefix's last symbol.
__device__ __forceinline__ uint32_t sample_walk(const OperandA &x, const SampleWalk &w,
                                                bool active, int32_t step, uint32_t *words,
                                                const DecodeTables *tb, int W, int rare) {
    uint32_t field = 0;
    if (step >= w.start) {
        field = tail_field(x.ov.tail[w.tail_index + (step - w.start)]);
    } else if (active) {
        StreamCursorT<kSampleGroup> cursor;
        cursor.init(words + threadIdx.x, tb, static_cast<uint32_t>(W), rare);
        for (int pair = 0; pair < step / 2; ++pair) {
            uint32_t f0, f1;
            cursor.advance(cursor.next_fields(f0, f1));
        }
        uint32_t f0, f1;
        cursor.next_fields(f0, f1);
        field = (step & 1) ? f1 : f0;
    }
    return join_entry(field, w.sm);
}

__global__ __launch_bounds__(kSampleGroup) void dual_sample_kernel(
    OperandA a, const uint16_t *__restrict__ a_samples, OperandA b,
    const uint16_t *__restrict__ b_samples, const float *__restrict__ alpha, int64_t n_blocks,
    int64_t logical_numel, int64_t sample_size, int S, int W, int rare,
    int32_t *__restrict__ partials, uint16_t *__restrict__ result_samples) {
    extern __shared__ uint32_t words[];   // A's then B's: 2 x (W + 1) rows x kSampleGroup
    __shared__ DecodeTables tba, tbb;
    const int t = threadIdx.x;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kSampleGroup + t;
    const bool active = i < sample_size;
    const int shift = __builtin_ctzll(static_cast<uint64_t>(sample_size));
    const int64_t pos = active ? sample_position(i, logical_numel, sample_size, shift) : 0;
    const int64_t row = pos / kLanes;
    const int32_t lane = static_cast<int32_t>((pos % kLanes) ^ (row & 254));
    const int64_t block = row >> (S == 128 ? 7 : 8);   // S is 128 or 256
    const int32_t step = static_cast<int32_t>(row & (S - 1));
    const bool walk_a = a_samples == nullptr, walk_b = b_samples == nullptr;
    uint32_t *words_a = words, *words_b = words + (W + 1) * kSampleGroup;
    SampleWalk wa{}, wb{};
    if (walk_a) {
        int32_t packed[256 / kSampleGroup];
#pragma unroll
        for (int k = 0; k < 256 / kSampleGroup; ++k)
            packed[k] = a.shifted_decode[t + k * kSampleGroup];
        sample_issue(a, active, row, lane, block, n_blocks, S, W, words_a, wa);
        const int32_t center = a.center[0];
#pragma unroll
        for (int k = 0; k < 256 / kSampleGroup; ++k)
            build_decode_entry(tba, t + k * kSampleGroup, packed[k], center);
    }
    if (walk_b) {
        int32_t packed[256 / kSampleGroup];
#pragma unroll
        for (int k = 0; k < 256 / kSampleGroup; ++k)
            packed[k] = b.shifted_decode[t + k * kSampleGroup];
        sample_issue(b, active, row, lane, block, n_blocks, S, W, words_b, wb);
        const int32_t center = b.center[0];
#pragma unroll
        for (int k = 0; k < 256 / kSampleGroup; ++k)
            build_decode_entry(tbb, t + k * kSampleGroup, packed[k], center);
    }
    wait_memory();
    __syncthreads();   // decode tables and staged words
    const uint32_t av = walk_a ? sample_walk(a, wa, active, step, words_a, &tba, W, rare)
                               : (active ? a_samples[i] : 0u);
    const uint32_t bv = walk_b ? sample_walk(b, wb, active, step, words_b, &tbb, W, rare)
                               : (active ? b_samples[i] : 0u);
    const uint32_t result =
        float_to_bf16(__builtin_fmaf(bf16_to_float(av), alpha[0], bf16_to_float(bv)));
    if (active && result_samples != nullptr) result_samples[i] = static_cast<uint16_t>(result);
    const int32_t exp = static_cast<int32_t>((result >> 7) & 255u) - 127;
    const bool keep = active && exp >= -120;
    const int32_t sum = wave_sum(keep ? exp : 0);
    const int32_t kept = wave_sum(keep ? 1 : 0);
    if (t == 0) {
        partials[2 * blockIdx.x] = sum;
        partials[2 * blockIdx.x + 1] = kept;
    }
}

// The two-operand kernel keeps its LDS to about 52 KiB at W = 25, so that
// three workgroups fit per CU and the C4-sized grid (688 codec blocks) runs
// in one round on 256 CUs:
//  * payload rows 0..2 of each stream live in registers (the cursor's initial
//    window) and only rows 3..W-1 are staged; past a stream's last word the
//    cursor re-reads word W-1 instead of a zero pad row (bits beyond a
//    stream's end never reach a decoded value);
//  * side bytes move in 8-step halves: each wave's 1 KiB slice holds A's half
//    (which the result's side bytes then overwrite) and B's half.
constexpr int kHalfSlice = kHalfSteps * kWave;   // one operand's 8-step half, one wave

using u32x2 = __attribute__((ext_vector_type(2))) uint32_t;

// This lane's 8 bytes of a wave's 8-step half: step j >> 3, lanes (j & 7) * 8..
// of the wave's 64 columns, so lane j's bytes land at j * 8 of the half.
__device__ __forceinline__ uint32_t half_side_offset() {
    const uint32_t j = threadIdx.x & (kWave - 1);
    const uint32_t wave = threadIdx.x / kWave;
    return (j >> 3) * kLanes + wave * kWave + (j & 7) * 8;
}

__device__ __forceinline__ u32x2 fetch_half_side(__amdgpu_buffer_rsrc_t side, uint32_t voffset,
                                                 int first_step) {
    return __builtin_amdgcn_raw_buffer_load_b64(side, voffset, first_step * kLanes, 0);
}

__device__ __forceinline__ void store_half_side(uint8_t *half, u32x2 q) {
    reinterpret_cast<u32x2 *>(half)[threadIdx.x & (kWave - 1)] = q;
}

// What a lane walks a block of two operands with (tails read from HBM).
struct DualWalk {
    QuadCursor ca, cb;
    LaneOverlay lane_a, lane_b;
    StreamWriter writer;
    const uint2 *enc;
    uint8_t *half_a, *half_b;   // this wave's 8 rows of side bytes of each operand
    float alpha;
    int64_t row_base;
    uint32_t valid;
};

// Emit the half at `first` from fa/fb while decoding the next half of both
// operands into them; the two operands' lookups are independent of each other
// and of the emitting.  kFast: every code is known to fit.
template <bool kFull, bool kFast>
__device__ __forceinline__ void dual_half_emit(DualWalk &u, uint32_t (&fa)[kHalfSteps],
                                               uint32_t (&fb)[kHalfSteps], const UpdateIo &io,
                                               int first, int S) {
    const uint32_t mask = static_cast<uint32_t>((u.row_base + first) & 254);
    Quad qa, qb;
    u.ca.first(qa);
    u.cb.first(qb);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t sa[kHalfSteps], sb[kHalfSteps];
#pragma unroll
    for (int k = 0; k < kHalfSteps; ++k) {
        sa[k] = side_byte(u.half_a, k);
        sb[k] = side_byte(u.half_b, k);
    }
    __builtin_amdgcn_sched_barrier(0);
    u.ca.second(qa);
    u.cb.second(qb);
    __builtin_amdgcn_sched_barrier(0);
    // fma(a, alpha, b) (pointwise_scalar_dual.py:226).
    float x[kHalfSteps];
#pragma unroll
    for (int k = 0; k < kHalfSteps; ++k)
        x[k] = __builtin_fmaf(__uint_as_float(join_float(fa[k], sa[k])), u.alpha,
                              __uint_as_float(join_float(fb[k], sb[k])));
    __builtin_amdgcn_sched_barrier(0);
    u.ca.third(qa);
    u.cb.third(qb);
    __builtin_amdgcn_sched_barrier(0);
    HalfEmit h;
    round_half<kFull>(h, x, first, mask, u.valid);
    store_half_sides(h, u.half_a);
    __builtin_amdgcn_sched_barrier(0);
    u.ca.fourth(qa);
    u.cb.fourth(qb);
    __builtin_amdgcn_sched_barrier(0);
    look_up_quad<kFull>(h, u.enc, 0, first, mask, u.valid);
    __builtin_amdgcn_sched_barrier(0);
    u.ca.finish(qa, fa);
    u.cb.finish(qb, fb);
    u.ca.first(qa);
    u.cb.first(qb);
    __builtin_amdgcn_sched_barrier(0);
    look_up_quad<kFull>(h, u.enc, 1, first, mask, u.valid);
    __builtin_amdgcn_sched_barrier(0);
    u.ca.second(qa);
    u.cb.second(qb);
    __builtin_amdgcn_sched_barrier(0);
    if (kFast) {
        const QuadCodes c0(h, 0), c1(h, 1);
        __builtin_amdgcn_sched_barrier(0);
        u.ca.third(qa);
        u.cb.third(qb);
        __builtin_amdgcn_sched_barrier(0);
        put_half(c0, c1, u.writer);
    } else {
        u.ca.third(qa);
        u.cb.third(qb);
        put_half_by_pairs(h, u.writer, first, mask, io.exponents);
    }
    __builtin_amdgcn_sched_barrier(0);
    u.ca.fourth(qa);
    u.cb.fourth(qb);
    u.ca.finish(qa, fa + 4);
    u.cb.finish(qb, fb + 4);
    overlay_half(u.lane_a, nullptr, first + kHalfSteps, S, fa);
    overlay_half(u.lane_b, nullptr, first + kHalfSteps, S, fb);
}

// The half at `first`, whose side bytes come in side_a/side_b; refills them with
// those of the half at first + 16 (two halves ahead: one half of work is far
// shorter than HBM's latency under load).
template <bool kFull>
__device__ __forceinline__ void dual_half(DualWalk &u, uint32_t (&fa)[kHalfSteps],
                                          uint32_t (&fb)[kHalfSteps], u32x2 &side_a,
                                          u32x2 &side_b, const UpdateIo &io, int first, int S) {
    const uint32_t voffset = half_side_offset();
    store_half_side(u.half_a, side_a);
    store_half_side(u.half_b, side_b);
    const int ahead = first + 2 * kHalfSteps;
    side_a = fetch_half_side(io.side, ahead < S ? voffset : kOutOfRange, ahead);
    side_b = fetch_half_side(io.other, ahead < S ? voffset : kOutOfRange, ahead);
    if (__builtin_expect(u.writer.fits_half(), 1))
        dual_half_emit<kFull, true>(u, fa, fb, io, first, S);
    else
        dual_half_emit<kFull, false>(u, fa, fb, io, first, S);
    // A's half now holds the result's side bytes.
    const u32x2 q = reinterpret_cast<const u32x2 *>(u.half_a)[threadIdx.x & (kWave - 1)];
    __builtin_amdgcn_raw_buffer_store_b64(q, io.side_out, voffset, first * kLanes, kSideStore);
}

// A whole block, with two copies of the prefetched side bytes as update_rows
// (io.other: B's side bytes).
template <bool kFull>
__device__ __forceinline__ void dual_rows(DualWalk &u, u32x2 side_a, u32x2 side_b,
                                          const UpdateIo &io, int S) {
    u32x2 next_a = fetch_half_side(io.side, half_side_offset(), kHalfSteps);
    u32x2 next_b = fetch_half_side(io.other, half_side_offset(), kHalfSteps);
    uint32_t fa[kHalfSteps], fb[kHalfSteps];
    u.ca.quad(fa);
    u.cb.quad(fb);
    u.ca.quad(fa + 4);
    u.cb.quad(fb + 4);
    overlay_half(u.lane_a, nullptr, 0, S, fa);
    overlay_half(u.lane_b, nullptr, 0, S, fb);
#pragma unroll 1
    for (int c = 0; c < S; c += 2 * kHalfSteps) {
        dual_half<kFull>(u, fa, fb, side_a, side_b, io, c, S);
        dual_half<kFull>(u, fa, fb, next_a, next_b, io, c + kHalfSteps, S);
    }
}

template <bool kBooked>
__global__ __launch_bounds__(kLanes) void dual_encode_kernel(
    OperandA a, OperandA b, const float *__restrict__ alpha,
    const int32_t *__restrict__ partials, int32_t n_groups,
    const int32_t *__restrict__ base_encode, const int32_t *__restrict__ base_decode,
    int32_t *__restrict__ center_out, int32_t *__restrict__ shifted_decode_out,
    uint8_t *__restrict__ side_out, int32_t *__restrict__ encoded_out,
    uint8_t *__restrict__ extra_starts, int32_t *__restrict__ summaries,
    uint8_t *__restrict__ exponents, int64_t n_blocks, int64_t logical_numel, int S, int W,
    int rare, KernelBookkeeping bk) {
    extern __shared__ uint32_t stages[];   // A's rows 3..W-1, then B's
    __shared__ QuadTables tba, tbb;
    __shared__ uint2 enc[256];
    __shared__ int32_t scratch[kWavesPerBlock];
    __shared__ int32_t shared_center[2];   // center, and whether its samples failed to arrive
    // The overflow maps (2 KiB) and the raw encode table (1 KiB) are only used
    // before the first side halves are stored, so they share the slices.
    __shared__ __attribute__((aligned(16))) uint8_t slices[kWavesPerBlock][2 * kHalfSlice];
    int32_t *map_start = reinterpret_cast<int32_t *>(&slices[0][0]);
    int32_t *map_offset = map_start + kLanes;
    int32_t *raw_encode = map_offset + kLanes;
    uint32_t *stage_a = stages;
    uint32_t *stage_b = stages + register_stage_bytes(W) / 4;
    const int t = threadIdx.x;
    const int64_t block = blockIdx.x;
    const bool sampled_here = kBooked && bk.sample_groups > 0;
    if (sampled_here && block < bk.sample_groups && t < kWave) {
        // fma(a, alpha, b) (pointwise_scalar_dual.py:226) at sample group
        // `block`'s positions from both operands' recorded values.
        const int64_t i = block * kSampleGroup + t;
        const bool active = i < bk.sample_size;
        uint32_t result = 0;
        if (active) {
            result = float_to_bf16(__builtin_fmaf(bf16_to_float(bk.a_samples[i]), alpha[0],
                                                  bf16_to_float(bk.b_samples[i])));
            if (bk.result_samples != nullptr)
                bk.result_samples[i] = static_cast<uint16_t>(result);
        }
        const int32_t exp = static_cast<int32_t>((result >> 7) & 255u) - 127;
        const bool keep = active && exp >= -120;
        const int32_t sum = wave_sum(keep ? exp : 0);
        const int32_t kept = wave_sum(keep ? 1 : 0);
        publish_sample_group(bk, block, sum, kept);
    }
    if (block >= n_blocks) return;   // a sample group past the last block
    const int64_t n_streams = n_blocks * kLanes;
    const int64_t row_base = block * S;
    const int64_t logical_base = row_base * kLanes;
    const uint32_t block_elems = static_cast<uint32_t>(S) * kLanes;
    const int64_t remaining = logical_numel - logical_base;
    const uint32_t valid = remaining < block_elems ? static_cast<uint32_t>(remaining) : block_elems;
    UpdateIo io;
    io.side = make_rsrc(a.side + logical_base, block_elems);
    io.other = make_rsrc(b.side + logical_base, block_elems);   // B's side bytes
    io.side_out = make_rsrc(side_out + logical_base, block_elems);
    io.exponents = make_rsrc(exponents + logical_base, valid);
    const u32x2 first_a = fetch_half_side(io.side, half_side_offset(), 0);
    const u32x2 first_b = fetch_half_side(io.other, half_side_offset(), 0);
    // Loads the prologue needs later, issued now so that they share one round
    // trip with the tables' loads instead of following its barriers.
    const OverlayHead head_a = load_overlay_head(a.ov, a.has_overlay != 0, block, n_blocks);
    const OverlayHead head_b = load_overlay_head(b.ov, b.has_overlay != 0, block, n_blocks);
    const BaseDecodeShare base0 = load_base_decode(base_decode, block == 0);
    const float alpha_value = alpha[0];
    // Each stream's first three words: the cursors' initial windows.
    uint32_t wa[kRegisterRows], wb[kRegisterRows];
    load_register_rows(a.encoded, n_streams, block, wa);
    load_register_rows(b.encoded, n_streams, block, wb);

    raw_encode[t] = base_encode[t];
    if (sampled_here) {
        center_from_control(bk.control, bk.sample_groups, bk.epoch, bk.polls, shared_center);
    } else {
        center_from_partials(partials, n_groups, shared_center);
        if (t == 0) shared_center[1] = 0;
    }
    build_quad_tables(tba, a.shifted_decode, rare);
    build_quad_tables(tbb, b.shifted_decode, rare);
    const int32_t a_center = a.center[0], b_center = b.center[0];
    stage_payload_rows(stage_a, a.encoded, n_streams, block, kRegisterRows, W);
    stage_payload_rows(stage_b, b.encoded, n_streams, block, kRegisterRows, W);
    __syncthreads();   // center and raw encode table
    const int32_t center = shared_center[0];
    const bool center_failed = shared_center[1] != 0;
    enc[t] = repack_encode_entry(static_cast<uint32_t>(raw_encode[byte_to_index(t, center)]));
    if (block == 0) {
        if (t == 0) center_out[0] = center;
        store_shifted_decode(shifted_decode_out, base0, center);
    }
    __syncthreads();   // raw_encode is no longer read (it shares the maps' LDS)
    const LaneOverlay lane_a = build_overlay(a.ov, head_a, S, map_start, map_offset, scratch,
                                             nullptr, 0);
    __syncthreads();   // B's overlay reuses the maps
    const LaneOverlay lane_b = build_overlay(b.ov, head_b, S, map_start, map_offset, scratch,
                                             nullptr, 0);
    wait_memory();
    __syncthreads();   // payloads and encode table visible; maps no longer read

    DualWalk u;
    u.ca.init(stage_a + t, &tba, static_cast<uint32_t>(W), rare, wa, a_center);
    u.cb.init(stage_b + t, &tbb, static_cast<uint32_t>(W), rare, wb, b_center);
    u.lane_a = lane_a;
    u.lane_b = lane_b;
    const uint32_t row_bytes = static_cast<uint32_t>(n_streams * 4);
    u.writer = StreamWriter{make_rsrc(encoded_out + block * kLanes,
                                      static_cast<uint32_t>(W - 1) * row_bytes + kLanes * 4),
                            row_bytes, static_cast<uint32_t>(t) * 4u,
                            static_cast<uint32_t>(W) * row_bytes + static_cast<uint32_t>(t) * 4u,
                            static_cast<uint32_t>(W) * 32u, 0u, 0u, 0u};
    u.writer.keep_row_bytes_in_vgpr();
    u.enc = enc;
    u.half_a = slices[t / kWave];
    u.half_b = u.half_a + kHalfSlice;
    u.alpha = alpha_value;
    u.row_base = row_base;
    u.valid = valid;
    if (valid == block_elems)
        dual_rows<true>(u, first_a, first_b, io, S);
    else
        dual_rows<false>(u, first_a, first_b, io, S);
    u.writer.finish();
    const bool overflow = u.writer.overflowed();
    const int32_t extra = u.writer.extra_start();
    extra_starts[block * kLanes + t] = static_cast<uint8_t>(overflow ? extra : 255);
    // Streams from bit 20 (at most 256), tail bytes in bits 0..19 (at most
    // 256 x 256): one block scan.
    const int32_t both = block_sum(overflow ? (S - extra) | (1 << 20) : 0, scratch);
    publish_block<kBooked>(bk, summaries, block, n_blocks, both >> 20, both & 0xFFFFF,
                           reinterpret_cast<int32_t *>(stages), map_start, SingleBook{},
                           center_failed);
}

int32_t check_operand(const int32_t *encoded, const uint8_t *side, const int32_t *shifted_decode,
                      const int32_t *center, const lct_overflow *overflow) {
    if (!encoded || !side || !shifted_decode || !center) return LCT_E_NULL;
    if (overflow != nullptr) {
        if (!overflow->lanes || !overflow->starts || !overflow->tail || !overflow->blocks)
            return LCT_E_NULL;
        if (overflow->descriptor != nullptr && overflow->count == nullptr) return LCT_E_NULL;
    }
    return LCT_OK;
}

int32_t check_op(int32_t op, int32_t alpha_is_one, int32_t beta_is_one, const float *alpha,
                 const float *beta) {
    if (op < LCT_OP_ADD || op > LCT_OP_SCALAR_MUL_ADD) return LCT_E_ARG;
    if (op == LCT_OP_SCALAR_MUL_ADD && ((!alpha_is_one && !alpha) || (!beta_is_one && !beta)))
        return LCT_E_NULL;
    return LCT_OK;
}

int32_t check_shape(int64_t size, int64_t logical_numel, const lct_geometry &g,
                    int32_t rare_length) {
    if (!geometry_ok(g)) return LCT_E_GEOMETRY;
    if (logical_numel <= 0 || size <= 0 || size % g.block_symbols != 0 || logical_numel > size
        || logical_numel <= size - g.block_symbols || size / g.block_symbols > kMaxBlocks)
        return LCT_E_SIZE;
    if (rare_length < 0 || rare_length > 8) return LCT_E_ARG;
    return LCT_OK;
}

int32_t check_samples(int64_t sample_size, int64_t logical_numel) {
    if (sample_size <= 0 || sample_size > kMaxSamples || sample_size > logical_numel)
        return LCT_E_SIZE;
    if (sample_size != logical_numel && (sample_size & (sample_size - 1)) != 0) return LCT_E_ARG;
    return LCT_OK;
}

}  // namespace
}  // namespace lct

using namespace lct;

extern "C" int32_t lct_pointwise_sample(const int32_t *encoded, const uint8_t *side,
                                        const int32_t *shifted_decode, const int32_t *center,
                                        const lct_overflow *overflow, const void *a_samples,
                                        const void *other, const float *alpha,
                                        const float *beta, int64_t size,
                                        int64_t logical_numel, lct_geometry g,
                                        int32_t rare_length, int32_t op, int32_t alpha_is_one,
                                        int32_t beta_is_one, int64_t sample_size,
                                        int32_t *partials, void *result_samples,
                                        hipStream_t stream) {
    if (int32_t e = check_operand(encoded, side, shifted_decode, center, overflow)) return e;
    if (!other || !partials) return LCT_E_NULL;
    if (int32_t e = check_op(op, alpha_is_one, beta_is_one, alpha, beta)) return e;
    if (int32_t e = check_shape(size, logical_numel, g, rare_length)) return e;
    if (int32_t e = check_samples(sample_size, logical_numel)) return e;
    const OperandA a{encoded, side, shifted_decode, center,
                     overflow ? *overflow : lct_overflow{}, overflow != nullptr};
    const OpArgs args{alpha, beta, op, alpha_is_one, beta_is_one};
    const int64_t n_blocks = size / g.block_symbols;
    const size_t lds = static_cast<size_t>(g.fixed_words + 1) * kSampleGroup * sizeof(uint32_t);
    hipLaunchKernelGGL(pointwise_sample_kernel, dim3(sample_groups(sample_size)),
                       dim3(kSampleGroup), lds, stream, a,
                       static_cast<const uint16_t *>(a_samples),
                       static_cast<const uint16_t *>(other), args, n_blocks, logical_numel,
                       sample_size, g.steps, g.fixed_words, rare_length, partials,
                       static_cast<uint16_t *>(result_samples));
    return static_cast<int32_t>(hipGetLastError());
}

namespace {

// The host side of lct_bookkeeping: validated against the launch's block
// count, in the kernel's form (bk.control == nullptr without one).  Also
// raises `lds` to the free list's LDS copy when buffered.
int32_t prepare_bookkeeping(const lct_bookkeeping *in, int64_t n_blocks, KernelBookkeeping &bk,
                            size_t &lds) {
    bk = KernelBookkeeping{};
    if (in == nullptr) return LCT_OK;
    if (!in->control || !in->counts || !in->blocks) return LCT_E_NULL;
    if (n_blocks > kMaxBlocks) return LCT_E_SIZE;
    if (in->control_words < kControlPartials + n_blocks) return LCT_E_SIZE;
    // Epoch 0 would match a control array's initial zeros.
    if (in->epoch == 0) return LCT_E_ARG;
    if ((reinterpret_cast<uintptr_t>(in->control) & 7) != 0) return LCT_E_ARG;
    if (in->buffer_meta != nullptr) {
        if (!in->descriptor) return LCT_E_NULL;
        if (in->max_free_regions <= 0 || in->max_free_regions > 4096
            || (in->max_free_regions & (in->max_free_regions - 1)) != 0)
            return LCT_E_ARG;
        if (in->frees.count < 0 || in->frees.count > LCT_MAX_PENDING_FREES) return LCT_E_ARG;
        for (int i = 0; i < in->frees.count; ++i)
            if (in->frees.descriptor[i] == nullptr) return LCT_E_NULL;
        const size_t list = static_cast<size_t>(in->max_free_regions) * 8;
        if (list > lds) lds = list;
    }
    bk.control = in->control;
    bk.epoch = in->epoch;
    bk.counts = in->counts;
    bk.blocks = in->blocks;
    bk.descriptor = in->buffer_meta != nullptr ? in->descriptor : nullptr;
    bk.buffer_meta = in->buffer_meta;
    bk.max_free_regions = in->max_free_regions;
    if (in->buffer_meta != nullptr) bk.frees = in->frees;
    bk.lock_spins = lock_spins();
    bk.polls = ready_polls();
    return LCT_OK;
}

int32_t launch_pointwise_encode(
    const int32_t *encoded, const uint8_t *side, const int32_t *shifted_decode,
    const int32_t *center, const lct_overflow *overflow, const void *other, const float *alpha,
    const float *beta, const int32_t *partials, int64_t sample_size, const int32_t *base_encode,
    const int32_t *base_decode, int32_t *center_out, int32_t *shifted_decode_out,
    uint8_t *side_out, int32_t *encoded_out, uint8_t *extra_starts, int32_t *summaries,
    uint8_t *exponents, int64_t size, int64_t logical_numel, lct_geometry g, int32_t rare_length,
    int32_t op, int32_t alpha_is_one, int32_t beta_is_one, const lct_bookkeeping *bookkeeping,
    hipStream_t stream) {
    if (int32_t e = check_operand(encoded, side, shifted_decode, center, overflow)) return e;
    if (!other || !partials || !base_encode || !base_decode || !center_out || !shifted_decode_out
        || !side_out || !encoded_out || !extra_starts || !summaries || !exponents)
        return LCT_E_NULL;
    if (int32_t e = check_op(op, alpha_is_one, beta_is_one, alpha, beta)) return e;
    if (int32_t e = check_shape(size, logical_numel, g, rare_length)) return e;
    if (int32_t e = check_samples(sample_size, logical_numel)) return e;
    // 16-byte accesses: A's payload staging, A's and the result's side bytes.
    if (((reinterpret_cast<uintptr_t>(encoded) | reinterpret_cast<uintptr_t>(side)
          | reinterpret_cast<uintptr_t>(side_out)) & 15) != 0)
        return LCT_E_ARG;
    const int64_t n_blocks = size / g.block_symbols;
    // The result's payload words are addressed with 32-bit buffer offsets.
    if (static_cast<int64_t>(g.fixed_words) * n_blocks * kLanes * 4 >= (int64_t{1} << 31))
        return LCT_E_SIZE;
    const OperandA a{encoded, side, shifted_decode, center,
                     overflow ? *overflow : lct_overflow{}, overflow != nullptr};
    const OpArgs args{alpha, beta, op, alpha_is_one, beta_is_one};
    const int32_t groups = sample_groups(sample_size);
    size_t lds = static_cast<size_t>(register_stage_bytes(g.fixed_words));
    KernelBookkeeping bk;
    if (int32_t e = prepare_bookkeeping(bookkeeping, n_blocks, bk, lds)) return e;
    const auto kernel = bk.control != nullptr ? pointwise_encode_kernel<true>
                                              : pointwise_encode_kernel<false>;
    if (hipError_t e = reserve_dynamic_lds(reinterpret_cast<const void *>(kernel), lds))
        return static_cast<int32_t>(e);
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(n_blocks)),
                       dim3(kLanes), lds, stream, a, static_cast<const uint16_t *>(other), args,
                       partials, groups, base_encode, base_decode, center_out,
                       shifted_decode_out, side_out, encoded_out, extra_starts, summaries,
                       exponents, n_blocks, logical_numel, g.steps, g.fixed_words, rare_length,
                       bk);
    return static_cast<int32_t>(hipGetLastError());
}

}  // namespace

extern "C" int32_t lct_pointwise_encode(
    const int32_t *encoded, const uint8_t *side, const int32_t *shifted_decode,
    const int32_t *center, const lct_overflow *overflow, const void *other, const float *alpha,
    const float *beta, const int32_t *partials, int64_t sample_size, const int32_t *base_encode,
    const int32_t *base_decode, int32_t *center_out, int32_t *shifted_decode_out,
    uint8_t *side_out, int32_t *encoded_out, uint8_t *extra_starts, int32_t *summaries,
    uint8_t *exponents, int64_t size, int64_t logical_numel, lct_geometry g, int32_t rare_length,
    int32_t op, int32_t alpha_is_one, int32_t beta_is_one, hipStream_t stream) {
    return launch_pointwise_encode(encoded, side, shifted_decode, center, overflow, other, alpha,
                                   beta, partials, sample_size, base_encode, base_decode,
                                   center_out, shifted_decode_out, side_out, encoded_out,
                                   extra_starts, summaries, exponents, size, logical_numel, g,
                                   rare_length, op, alpha_is_one, beta_is_one, nullptr, stream);
}

extern "C" int32_t lct_pointwise_encode_fused(
    const int32_t *encoded, const uint8_t *side, const int32_t *shifted_decode,
    const int32_t *center, const lct_overflow *overflow, const void *other, const float *alpha,
    const float *beta, const int32_t *partials, int64_t sample_size, const int32_t *base_encode,
    const int32_t *base_decode, int32_t *center_out, int32_t *shifted_decode_out,
    uint8_t *side_out, int32_t *encoded_out, uint8_t *extra_starts, int32_t *summaries,
    uint8_t *exponents, int64_t size, int64_t logical_numel, lct_geometry g, int32_t rare_length,
    int32_t op, int32_t alpha_is_one, int32_t beta_is_one, const lct_bookkeeping *bookkeeping,
    hipStream_t stream) {
    if (!bookkeeping) return LCT_E_NULL;
    return launch_pointwise_encode(encoded, side, shifted_decode, center, overflow, other, alpha,
                                   beta, partials, sample_size, base_encode, base_decode,
                                   center_out, shifted_decode_out, side_out, encoded_out,
                                   extra_starts, summaries, exponents, size, logical_numel, g,
                                   rare_length, op, alpha_is_one, beta_is_one, bookkeeping,
                                   stream);
}

extern "C" int32_t lct_dual_sample(const int32_t *a_encoded, const uint8_t *a_side,
                                   const int32_t *a_shifted_decode, const int32_t *a_center,
                                   const lct_overflow *a_overflow, const void *a_samples,
                                   const int32_t *b_encoded, const uint8_t *b_side,
                                   const int32_t *b_shifted_decode, const int32_t *b_center,
                                   const lct_overflow *b_overflow, const void *b_samples,
                                   const float *alpha, int64_t size, int64_t logical_numel,
                                   lct_geometry g, int32_t rare_length, int64_t sample_size,
                                   int32_t *partials, void *result_samples,
                                   hipStream_t stream) {
    if (int32_t e = check_operand(a_encoded, a_side, a_shifted_decode, a_center, a_overflow))
        return e;
    if (int32_t e = check_operand(b_encoded, b_side, b_shifted_decode, b_center, b_overflow))
        return e;
    if (!alpha || !partials) return LCT_E_NULL;
    if (int32_t e = check_shape(size, logical_numel, g, rare_length)) return e;
    if (int32_t e = check_samples(sample_size, logical_numel)) return e;
    const OperandA a{a_encoded, a_side, a_shifted_decode, a_center,
                     a_overflow ? *a_overflow : lct_overflow{}, a_overflow != nullptr};
    const OperandA b{b_encoded, b_side, b_shifted_decode, b_center,
                     b_overflow ? *b_overflow : lct_overflow{}, b_overflow != nullptr};
    const int64_t n_blocks = size / g.block_symbols;
    const size_t lds = 2 * static_cast<size_t>(g.fixed_words + 1) * kSampleGroup * sizeof(uint32_t);
    hipLaunchKernelGGL(dual_sample_kernel, dim3(sample_groups(sample_size)), dim3(kSampleGroup),
                       lds, stream, a, static_cast<const uint16_t *>(a_samples), b,
                       static_cast<const uint16_t *>(b_samples), alpha, n_blocks, logical_numel,
                       sample_size, g.steps, g.fixed_words, rare_length, partials,
                       static_cast<uint16_t *>(result_samples));
    return static_cast<int32_t>(hipGetLastError());
}

namespace {

int32_t launch_dual_encode(
    const int32_t *a_encoded, const uint8_t *a_side, const int32_t *a_shifted_decode,
    const int32_t *a_center, const lct_overflow *a_overflow, const int32_t *b_encoded,
    const uint8_t *b_side, const int32_t *b_shifted_decode, const int32_t *b_center,
    const lct_overflow *b_overflow, const float *alpha, const int32_t *partials,
    int64_t sample_size, const int32_t *base_encode, const int32_t *base_decode,
    int32_t *center_out, int32_t *shifted_decode_out, uint8_t *side_out, int32_t *encoded_out,
    uint8_t *extra_starts, int32_t *summaries, uint8_t *exponents, int64_t size,
    int64_t logical_numel, lct_geometry g, int32_t rare_length,
    const lct_bookkeeping *bookkeeping, hipStream_t stream) {
    if (int32_t e = check_operand(a_encoded, a_side, a_shifted_decode, a_center, a_overflow))
        return e;
    if (int32_t e = check_operand(b_encoded, b_side, b_shifted_decode, b_center, b_overflow))
        return e;
    // With both operands' recorded sample values the launch samples the center.
    const bool sample_here = bookkeeping != nullptr && bookkeeping->a_samples != nullptr
        && bookkeeping->b_samples != nullptr;
    if (!alpha || (!partials && !sample_here) || !base_encode || !base_decode || !center_out
        || !shifted_decode_out || !side_out || !encoded_out || !extra_starts || !summaries
        || !exponents)
        return LCT_E_NULL;
    if (int32_t e = check_shape(size, logical_numel, g, rare_length)) return e;
    if (int32_t e = check_samples(sample_size, logical_numel)) return e;
    // 16-byte accesses: payload staging, A's, B's and the result's side bytes.
    if (((reinterpret_cast<uintptr_t>(a_encoded) | reinterpret_cast<uintptr_t>(b_encoded)
          | reinterpret_cast<uintptr_t>(a_side) | reinterpret_cast<uintptr_t>(b_side)
          | reinterpret_cast<uintptr_t>(side_out)) & 15) != 0)
        return LCT_E_ARG;
    const int64_t n_blocks = size / g.block_symbols;
    // The result's payload words are addressed with 32-bit buffer offsets.
    if (static_cast<int64_t>(g.fixed_words) * n_blocks * kLanes * 4 >= (int64_t{1} << 31))
        return LCT_E_SIZE;
    const OperandA a{a_encoded, a_side, a_shifted_decode, a_center,
                     a_overflow ? *a_overflow : lct_overflow{}, a_overflow != nullptr};
    const OperandA b{b_encoded, b_side, b_shifted_decode, b_center,
                     b_overflow ? *b_overflow : lct_overflow{}, b_overflow != nullptr};
    // Rows 0..2 of every stream start in registers (W = 2 or 3 never occurs in
    // a reference geometry).
    if (g.fixed_words <= kRegisterRows) return LCT_E_GEOMETRY;
    size_t lds = 2 * static_cast<size_t>(register_stage_bytes(g.fixed_words));
    KernelBookkeeping bk;
    if (int32_t e = prepare_bookkeeping(bookkeeping, n_blocks, bk, lds)) return e;
    int64_t grid = n_blocks;
    if (sample_here) {
        bk.a_samples = bookkeeping->a_samples;
        bk.b_samples = bookkeeping->b_samples;
        bk.result_samples = bookkeeping->result_samples;
        bk.sample_size = sample_size;
        bk.sample_groups = sample_groups(sample_size);
        grid = std::max<int64_t>(n_blocks, bk.sample_groups);
    }
    const auto kernel = bk.control != nullptr ? dual_encode_kernel<true>
                                              : dual_encode_kernel<false>;
    if (hipError_t e = reserve_dynamic_lds(reinterpret_cast<const void *>(kernel), lds))
        return static_cast<int32_t>(e);
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(grid)), dim3(kLanes),
                       lds, stream, a, b, alpha, partials, sample_groups(sample_size),
                       base_encode, base_decode, center_out, shifted_decode_out, side_out,
                       encoded_out, extra_starts, summaries, exponents, n_blocks, logical_numel,
                       g.steps, g.fixed_words, rare_length, bk);
    return static_cast<int32_t>(hipGetLastError());
}

}  // namespace

extern "C" int32_t lct_dual_encode(
    const int32_t *a_encoded, const uint8_t *a_side, const int32_t *a_shifted_decode,
    const int32_t *a_center, const lct_overflow *a_overflow, const int32_t *b_encoded,
    const uint8_t *b_side, const int32_t *b_shifted_decode, const int32_t *b_center,
    const lct_overflow *b_overflow, const float *alpha, const int32_t *partials,
    int64_t sample_size, const int32_t *base_encode, const int32_t *base_decode,
    int32_t *center_out, int32_t *shifted_decode_out, uint8_t *side_out, int32_t *encoded_out,
    uint8_t *extra_starts, int32_t *summaries, uint8_t *exponents, int64_t size,
    int64_t logical_numel, lct_geometry g, int32_t rare_length, hipStream_t stream) {
    return launch_dual_encode(a_encoded, a_side, a_shifted_decode, a_center, a_overflow,
                              b_encoded, b_side, b_shifted_decode, b_center, b_overflow, alpha,
                              partials, sample_size, base_encode, base_decode, center_out,
                              shifted_decode_out, side_out, encoded_out, extra_starts, summaries,
                              exponents, size, logical_numel, g, rare_length, nullptr, stream);
}

extern "C" int32_t lct_dual_encode_fused(
    const int32_t *a_encoded, const uint8_t *a_side, const int32_t *a_shifted_decode,
    const int32_t *a_center, const lct_overflow *a_overflow, const int32_t *b_encoded,
    const uint8_t *b_side, const int32_t *b_shifted_decode, const int32_t *b_center,
    const lct_overflow *b_overflow, const float *alpha, const int32_t *partials,
    int64_t sample_size, const int32_t *base_encode, const int32_t *base_decode,
    int32_t *center_out, int32_t *shifted_decode_out, uint8_t *side_out, int32_t *encoded_out,
    uint8_t *extra_starts, int32_t *summaries, uint8_t *exponents, int64_t size,
    int64_t logical_numel, lct_geometry g, int32_t rare_length,
    const lct_bookkeeping *bookkeeping, hipStream_t stream) {
    if (!bookkeeping) return LCT_E_NULL;
    return launch_dual_encode(a_encoded, a_side, a_shifted_decode, a_center, a_overflow,
                              b_encoded, b_side, b_shifted_decode, b_center, b_overflow, alpha,
                              partials, sample_size, base_encode, base_decode, center_out,
                              shifted_decode_out, side_out, encoded_out, extra_starts, summaries,
                              exponents, size, logical_numel, g, rare_length, bookkeeping,
                              stream);
}

extern "C" int32_t lct_pointwise_update_batch(
    const lct_update_job *jobs, int32_t n_jobs, int32_t op, int32_t alpha_is_one,
    int32_t beta_is_one, const float *alpha, const float *beta, int32_t *partials,
    int64_t partial_words, uint8_t *extra_starts, int64_t extra_bytes, int32_t *summaries,
    int64_t summary_words, uint64_t *control, int64_t control_words, uint32_t epoch,
    int32_t *buffer_meta, int32_t max_free_regions, uint8_t *arena,
    const lct_pending_frees *frees, hipStream_t stream) {
    if (!jobs || !partials || !extra_starts || !summaries || !control || !buffer_meta || !arena)
        return LCT_E_NULL;
    if (n_jobs <= 0 || n_jobs > LCT_MAX_UPDATE_BATCH) return LCT_E_ARG;
    if (int32_t e = check_op(op, alpha_is_one, beta_is_one, alpha, beta)) return e;
    if (epoch == 0 || (reinterpret_cast<uintptr_t>(control) & 7) != 0) return LCT_E_ARG;
    if (max_free_regions <= 0 || max_free_regions > 4096
        || (max_free_regions & (max_free_regions - 1)) != 0)
        return LCT_E_ARG;
    UpdateSampleBatch sample{};
    UpdateEncodeBatch encode{};
    CompactBatch compact{};
    sample.n_jobs = encode.n_jobs = compact.n_jobs = n_jobs;
    sample.args = encode.args = OpArgs{alpha, beta, op, alpha_is_one, beta_is_one};
    encode.buffer_meta = buffer_meta;
    encode.max_free_regions = max_free_regions;
    if (frees != nullptr) {
        if (frees->count < 0 || frees->count > LCT_MAX_PENDING_FREES) return LCT_E_ARG;
        for (int i = 0; i < frees->count; ++i)
            if (frees->descriptor[i] == nullptr) return LCT_E_NULL;
        encode.frees = *frees;
    }
    encode.epoch = epoch;
    encode.lock_spins = lock_spins();
    encode.polls = ready_polls();
    static_assert(LCT_MAX_UPDATE_BATCH <= kMaxBatchJobs, "a request slot per job");
    compact.arena = arena;
    compact.steps = 0;
    compact.precomputed = 1;
    int64_t groups = 0, blocks_total = 0, partial_used = 0, extra_used = 0, summary_used = 0,
            control_used = 1;
    int max_words = 0;
    for (int j = 0; j < n_jobs; ++j) {
        const lct_update_job &in = jobs[j];
        const lct_geometry &g = in.geometry;
        const lct_overflow *ov = in.has_overflow ? &in.overflow : nullptr;
        if (int32_t e = check_operand(in.encoded, in.side, in.shifted_decode, in.center, ov))
            return e;
        if (!in.other || !in.base_encode || !in.base_decode || !in.center_out
            || !in.shifted_decode_out || !in.side_out || !in.encoded_out || !in.exponents
            || !in.counts || !in.blocks || !in.descriptor)
            return LCT_E_NULL;
        if (int32_t e = check_shape(in.size, in.logical_numel, g, in.rare_length)) return e;
        if (int32_t e = check_samples(in.sample_size, in.logical_numel)) return e;
        if (((reinterpret_cast<uintptr_t>(in.encoded) | reinterpret_cast<uintptr_t>(in.side)
              | reinterpret_cast<uintptr_t>(in.side_out)) & 15) != 0)
            return LCT_E_ARG;
        const int64_t nb = in.size / g.block_symbols;
        if (static_cast<int64_t>(g.fixed_words) * nb * kLanes * 4 >= (int64_t{1} << 31))
            return LCT_E_SIZE;
        // The compaction launch takes one step count for all its jobs.
        if (compact.steps != 0 && compact.steps != g.steps) return LCT_E_ARG;
        compact.steps = g.steps;
        const int32_t n_groups = sample_groups(in.sample_size);
        const OperandA a{in.encoded, in.side, in.shifted_decode, in.center,
                         ov ? *ov : lct_overflow{}, ov != nullptr};
        UpdateSampleJob &sj = sample.jobs[j];
        sj.a = a;
        sj.a_samples = static_cast<const uint16_t *>(in.a_samples);
        sj.other = static_cast<const uint16_t *>(in.other);
        sj.partials = partials + partial_used;
        sj.result_samples = static_cast<uint16_t *>(in.result_samples);
        sj.n_blocks = nb;
        sj.logical_numel = in.logical_numel;
        sj.sample_size = in.sample_size;
        sj.steps = g.steps;
        sj.fixed_words = g.fixed_words;
        sj.rare = in.rare_length;
        UpdateEncodeJob &ej = encode.jobs[j];
        ej.a = a;
        ej.other = sj.other;
        ej.partials = sj.partials;
        ej.base_encode = in.base_encode;
        ej.base_decode = in.base_decode;
        ej.center_out = in.center_out;
        ej.shifted_decode_out = in.shifted_decode_out;
        ej.side_out = in.side_out;
        ej.encoded_out = in.encoded_out;
        ej.extra_starts = extra_starts + extra_used;
        ej.summaries = summaries + summary_used;
        ej.exponents = in.exponents;
        ej.control = control + control_used;
        ej.counts = in.counts;
        ej.blocks = in.blocks;
        ej.descriptor = in.descriptor;
        ej.n_blocks = nb;
        ej.logical_numel = in.logical_numel;
        ej.n_groups = n_groups;
        ej.steps = g.steps;
        ej.fixed_words = g.fixed_words;
        ej.rare = in.rare_length;
        CompactBatchJob &cj = compact.jobs[j];
        cj.source = in.exponents;
        cj.blocks = in.blocks;
        cj.counts = in.counts;
        cj.descriptor = in.descriptor;
        cj.extra_starts = ej.extra_starts;
        cj.n_blocks = nb;
        cj.logical_numel = in.logical_numel;
        sample.first_group[j] = static_cast<int32_t>(groups);
        encode.first_block[j] = compact.first_block[j] = static_cast<int32_t>(blocks_total);
        groups += n_groups;
        blocks_total += nb;
        partial_used += 2 * n_groups;
        extra_used += nb * kLanes;
        summary_used += 5 * nb + 1;
        control_used += kControlPartials + nb;
        if (g.fixed_words > max_words) max_words = g.fixed_words;
    }
    if (partial_used > partial_words || extra_used > extra_bytes
        || summary_used > summary_words || control_used > control_words)
        return LCT_E_SIZE;
    if (blocks_total > 0x7FFFFFFF) return LCT_E_SIZE;
    sample.first_group[n_jobs] = static_cast<int32_t>(groups);
    encode.first_block[n_jobs] = compact.first_block[n_jobs] = static_cast<int32_t>(blocks_total);

    const size_t sample_lds = static_cast<size_t>(max_words + 1) * kSampleGroup * 4;
    hipLaunchKernelGGL(pointwise_sample_batch_kernel, dim3(static_cast<uint32_t>(groups)),
                       dim3(kSampleGroup), sample_lds, stream, sample);
    if (hipError_t e = hipGetLastError()) return static_cast<int32_t>(e);
    const size_t encode_lds = std::max(static_cast<size_t>(register_stage_bytes(max_words)),
                                       static_cast<size_t>(max_free_regions) * 8);
    if (hipError_t e = reserve_dynamic_lds(
            reinterpret_cast<const void *>(&pointwise_encode_batch_kernel), encode_lds))
        return static_cast<int32_t>(e);
    hipLaunchKernelGGL(pointwise_encode_batch_kernel, dim3(static_cast<uint32_t>(blocks_total)),
                       dim3(kLanes), encode_lds, stream, encode);
    if (hipError_t e = hipGetLastError()) return static_cast<int32_t>(e);
    return static_cast<int32_t>(
        launch_compact_batch(compact, static_cast<uint32_t>(blocks_total), stream));
}
