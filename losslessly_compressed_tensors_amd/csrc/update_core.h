// Streams of the fused update kernels (gfx950): decoding four symbols per
// window and appending four codes at a time.
//
// The kernels are bounded by the instructions their few waves issue (2.7 waves
// per SIMD at 688 codec blocks) and by the waits between dependent LDS
// lookups, so both directions work in quads: one 32-bit window serves four
// lookups (direct codes are at most 8 bits, LCT/compression/huffman_tables.py:
// 106-107) and one window advance, and four codes of at most 32 bits together
// leave with one word update and one store.  What does not fit a quad (an
// escape, codes of more than 32 bits, the end of a stream) is found by one
// wave-uniform test per quad, after the fact.
#pragma once

#include "pointwise_ops.h"

namespace lct {

// Decode entries with the exponent in FP32 position: the code's length in
// bits 0..4, kEscapeFlag for an escape (whose length then includes the 8-bit
// literal), the exponent from bit 23, so a decoded value is one bit-field
// insert away from its FP32 bits (join_float).  Four entries' lengths (64 at
// most) and flags add up in bits 0..6 and 8..10.
constexpr uint32_t kEscapeFlag = 1u << 8;
constexpr uint32_t kQuadCheck = 0x77Fu;   // the sum's lengths and flags

struct QuadTables {
    uint32_t entry[256];
};

// One entry per thread of a 256-thread block.
__device__ __forceinline__ void build_quad_tables(QuadTables &tb,
                                                  const int32_t *__restrict__ shifted_decode,
                                                  int32_t rare) {
    const int32_t packed = shifted_decode[threadIdx.x];
    const int32_t length = packed & 255;
    const uint32_t field = static_cast<uint32_t>(((packed >> 8) + 127) & 255) << 23;
    tb.entry[threadIdx.x] = (length >= 1 && length <= 8)
                                ? (static_cast<uint32_t>(length) | field)
                                : (static_cast<uint32_t>(rare + 8) | kEscapeFlag);
}

// Exponent field of an overflow tail byte int8(e - 127).
__device__ __forceinline__ uint32_t tail_entry(uint32_t byte) {
    return ((byte + 127u) & 255u) << 23;
}

// Values loaded on a rare path, waited for there: where the paths meet, the
// compiler would otherwise make the common path wait for its own loads and
// stores in flight as well.
__device__ __forceinline__ void settle(uint32_t &v0, uint32_t &v1, uint32_t &v2, uint32_t &v3) {
    asm volatile("" : "+v"(v0), "+v"(v1), "+v"(v2), "+v"(v3));
}

// A quad being decoded: its window and its entries so far; o1..o3 are running
// sums of entries, whose low bits are the next symbol's offset.
struct Quad {
    uint32_t bits, t0, t1, t2, t3, o2, o3;
};

// One lane's stream: words w, w+1, w+2 in lo, hi, nx (the first three start
// there; rows 3..W-1 are staged, row r at stage[r * kLanes]), pos the bit
// offset in lo.  A quad consumes at most 32 bits, so it crosses at most one
// word.  Past the last word the window re-reads word W-1: bits beyond a
// stream's end never reach a decoded value.  A lane past its overflow start or
// past the tensor's end walks on through such bits; its rows are then
// replaced (overlay_half) or masked.
struct QuadCursor {
    const uint32_t *stage;
    const QuadTables *tb;
    uint32_t pos, lo, hi, nx, next_row, pad_row, pending;
    int32_t rare, center;

    __device__ __forceinline__ void init(const uint32_t *stage_rows, const QuadTables *tables,
                                         uint32_t words, int32_t rare_length,
                                         const uint32_t (&w)[kRegisterRows],
                                         int32_t center_value) {
        stage = stage_rows - kRegisterRows * kLanes;
        tb = tables;
        pos = 0;
        lo = w[0];
        hi = w[1];
        nx = w[2];
        next_row = kRegisterRows;
        pad_row = words - 1;
        pending = 0;
        rare = rare_length;
        center = center_value;
    }

    // The four lookups, one call each so that callers put independent work
    // between them.
    __device__ __forceinline__ void first(Quad &q) {
        pending = stage[next_row * kLanes];
        q.bits = __builtin_amdgcn_alignbit(hi, lo, pos);
        q.t0 = tb->entry[q.bits & 255u];
    }
    __device__ __forceinline__ void second(Quad &q) const {
        q.t1 = tb->entry[__builtin_amdgcn_ubfe(q.bits, q.t0, 8)];
    }
    __device__ __forceinline__ void third(Quad &q) const {
        q.o2 = q.t0 + q.t1;
        q.t2 = tb->entry[__builtin_amdgcn_ubfe(q.bits, q.o2, 8)];
    }
    __device__ __forceinline__ void fourth(Quad &q) const {
        q.o3 = q.o2 + q.t2;
        q.t3 = tb->entry[__builtin_amdgcn_ubfe(q.bits, q.o3, 8)];
    }

    // The entries into f[0..3], and past them.  A quad whose lengths add up to
    // at most 32 read only bits of its window; more (escapes or several long
    // codes) is decoded again as two pairs.
    __device__ __forceinline__ void finish(Quad &q, uint32_t *f) {
        uint32_t sum = q.o3 + q.t3;
        if (__builtin_expect(__any((sum & kQuadCheck) > 32u), 0)) {
            if (__any((sum & 127u) > 32u)) {
                sum = pair(q.t0, q.t1);
                advance(sum);
                sum = pair(q.t2, q.t3);
            } else {
                const uint32_t o1 = q.t0;
                q.t0 = escaped(q.bits, 0u, q.t0);
                q.t1 = escaped(q.bits, o1, q.t1);
                q.t2 = escaped(q.bits, q.o2, q.t2);
                q.t3 = escaped(q.bits, q.o3, q.t3);
            }
            settle(q.t0, q.t1, q.t2, q.t3);
            asm volatile("" : "+v"(pending));
        }
        f[0] = q.t0;
        f[1] = q.t1;
        f[2] = q.t2;
        f[3] = q.t3;
        advance(sum & 127u);
    }

    __device__ __forceinline__ void quad(uint32_t *f) {
        Quad q;
        first(q);
        second(q);
        third(q);
        fourth(q);
        finish(q, f);
    }

    // The entry at bit `offset` (low 5 bits) of `window`, with an escape's
    // exponent taken from its 8-bit literal table index (primitives.py:29-35).
    __device__ __forceinline__ uint32_t escaped(uint32_t window, uint32_t offset,
                                                uint32_t entry) const {
        const uint32_t literal =
            __builtin_amdgcn_ubfe(window, (offset & 31u) + static_cast<uint32_t>(rare), 8);
        const uint32_t exponent = static_cast<uint32_t>(
            (index_to_exponent(static_cast<int32_t>(literal), center) + 127) & 255);
        return (entry & kEscapeFlag) != 0 ? (entry & 31u) | (exponent << 23) : entry;
    }

    __device__ __forceinline__ uint32_t pair(uint32_t &t0, uint32_t &t1) {
        pending = stage[next_row * kLanes];
        const uint32_t bits = __builtin_amdgcn_alignbit(hi, lo, pos);
        t0 = tb->entry[bits & 255u];
        t1 = tb->entry[__builtin_amdgcn_ubfe(bits, t0, 8)];
        const uint32_t offset = t0;
        t0 = escaped(bits, 0u, t0);
        t1 = escaped(bits, offset, t1);
        return (t0 + t1) & 127u;
    }

    // Consume `bits` (at most 32).
    __device__ __forceinline__ void advance(uint32_t bits) {
        const uint32_t p = pos + bits;
        const bool cross = p >= 32u;
        pos = p & 31u;
        lo = cross ? hi : lo;
        hi = cross ? nx : hi;
        nx = cross ? pending : nx;
        next_row = cross ? min(next_row + 1u, pad_row) : next_row;
    }
};

// Rows of the half at `first` at or past this lane's overflow start take their
// exponents from its tail.  (The half past the block's last step, which the
// last half decodes for nothing, has no tail bytes.)
__device__ __forceinline__ void overlay_half(const LaneOverlay &lane, const uint8_t *tail_lds,
                                             int first, int S, uint32_t (&f)[kHalfSteps]) {
    if (__builtin_expect(lane.wave_start >= min(first + kHalfSteps, S), 1)) return;   // uniform
    if (first >= S) return;
#pragma unroll
    for (int j = 0; j < kHalfSteps; ++j) {
        if (first + j >= lane.start) {
            const int32_t i = lane.offset + (first + j - lane.start);
            f[j] = tail_entry(lane.lds ? tail_lds[i] : lane.tail[i]);
        }
    }
    settle(f[0], f[1], f[2], f[3]);
    settle(f[4], f[5], f[6], f[7]);
}

// Encoder state of one lane's output stream.  Word r of the stream is at byte
// r * row_bytes + 4 * lane of the block's payload resource.  pos counts the
// bits of every pair so far, so once a pair does not fit, pos stays above the
// limit and every later pair overflows too (encode.py:73-90: only the first
// overflowing pair matters); word and row_off then keep the bits before that
// pair, which finish() stores.
struct StreamWriter {
    __amdgpu_buffer_rsrc_t out;
    uint32_t row_bytes;   // 4 * n_streams
    uint32_t row_off;     // byte offset of the word being filled
    uint32_t end_off;     // row_off of row W
    uint32_t limit;       // 32 W
    uint32_t pos;         // bits of all pairs so far
    uint32_t word;        // bits of the word being filled
    uint32_t fits;        // pairs that fit

    __device__ __forceinline__ bool overflowed() const { return pos > limit; }

    // Hold row_bytes in a VGPR from here on: a row advance is then one
    // v_cndmask and one v_add (with row_bytes in an SGPR beside the SGPR
    // condition, gfx9's one-scalar-operand limit costs a copy each time).
    __device__ __forceinline__ void keep_row_bytes_in_vgpr() { asm volatile("" : "+v"(row_bytes)); }

    // The first pair that did not fit is the one after the pairs that fit, so
    // its (even) step is twice their count.
    __device__ __forceinline__ int32_t extra_start() const { return static_cast<int32_t>(2 * fits); }

    // Append the pair code of encode entries e0/e1 ({reversed code, length};
    // {0, 0} = no code), following encode.py:66-90.  Returns whether the pair
    // (and so every later one) overflows.  A pair that completes a word
    // stores it.
    __device__ __forceinline__ bool put(uint2 e0, uint2 e1) {
        const uint32_t code = e0.x | (e1.x << e0.y);
        const uint32_t len = e0.y + e1.y;
        const uint32_t shift = pos & 31u;
        const uint64_t placed = static_cast<uint64_t>(code) << shift;
        const uint32_t new_word = word | static_cast<uint32_t>(placed);
        const uint32_t after = pos + len;
        const bool ok = after <= limit;
        const bool completes = ok && shift + len >= 32u;
        __builtin_amdgcn_raw_buffer_store_b32(new_word, out, completes ? row_off : kOutOfRange,
                                              0, 0);
        row_off += completes ? row_bytes : 0u;
        word = ok ? (completes ? static_cast<uint32_t>(placed >> 32) : new_word) : word;
        fits += ok ? 1u : 0u;
        pos = after;
        return !ok;
    }

    // Append `len` <= 32 bits that are known to fit; the caller counts the
    // pairs.
    __device__ __forceinline__ void put_bits(uint32_t code, uint32_t len) {
        const uint32_t shift = pos & 31u;
        const uint64_t placed = static_cast<uint64_t>(code) << shift;
        const uint32_t new_word = word | static_cast<uint32_t>(placed);
        const bool completes = shift + len >= 32u;
        __builtin_amdgcn_raw_buffer_store_b32(new_word, out, completes ? row_off : kOutOfRange,
                                              0, 0);
        row_off += completes ? row_bytes : 0u;
        word = completes ? static_cast<uint32_t>(placed >> 32) : new_word;
        pos += len;
    }

    // Whether every pair of the next half fits for every lane of the wave (a
    // symbol's code is at most 16 bits: ESC of at most 8 bits and an 8-bit
    // literal).  Wave-uniform.
    __device__ __forceinline__ bool fits_half() const {
        return __all(pos + 16u * kHalfSteps <= limit);
    }

    // After the last pair: the word being filled (the bits before the first
    // pair that did not fit, for an overflowing stream), then zero words up to
    // row W-1.
    __device__ __forceinline__ void finish() {
        for (; row_off < end_off; row_off += row_bytes) {
            __builtin_amdgcn_raw_buffer_store_b32(word, out, row_off, 0, 0);
            word = 0u;
        }
    }
};

// Encode-table entry as the kernels keep it in LDS: {reversed code (<= 16
// bits), code length}, 8 bytes, so one 8-byte read gives both without masks
// (shifted tables: tables.py:53-67).
__device__ __forceinline__ uint2 repack_encode_entry(uint32_t packed) {
    return make_uint2(packed & 0xFFFFu, packed >> 20);
}

// Exponent bytes of a pair of BF16 results r (step s0 in bits 0..15, s0 + 1 in
// bits 16..31): bytes 0 and 2 of r >> 7.  The shift is kept opaque so that
// each encode-table address is one byte-selecting shift (SDWA) of it, where
// the compiler would otherwise fold shift and mask into two ops per index.
__device__ __forceinline__ uint32_t exponent_bytes(uint32_t r) {
    uint32_t x = r >> 7;
    asm("" : "+v"(x));
    return x;
}

// The results of one half (8 steps) of this lane's stream, two rows per word
// (step 2p in the low half of r[p]), from their FP32 values: rounded to BF16,
// and 0 (side byte 0, no code) at positions past the tensor's end (!kFull;
// off0: the half's first row's element offset within the block).
struct HalfEmit {
    uint32_t r[kHalfSteps / 2];
    uint2 e[kHalfSteps];   // their encode entries
};

// Element offset within the block of this lane's column in row `step`; mask
// is the swizzle mask of the half's first row, s0 the row's index in the half
// (even; the odd row after it is kLanes further).
__device__ __forceinline__ uint32_t half_offset(int first, uint32_t mask, int s0) {
    return static_cast<uint32_t>(first + s0) * kLanes
        + (threadIdx.x ^ mask ^ static_cast<uint32_t>(s0));
}

template <bool kFull>
__device__ __forceinline__ void round_half(HalfEmit &h, const float (&x)[kHalfSteps], int first,
                                           uint32_t mask, uint32_t valid) {
    uint64_t nan = 0;   // lanes with a NaN, kept in scalar registers
#pragma unroll
    for (int p = 0; p < kHalfSteps / 2; ++p) {
        const lct_f32x2 v = {x[2 * p], x[2 * p + 1]};
        h.r[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, lct_bf16x2));
        nan |= __builtin_amdgcn_ballot_w64(__builtin_isunordered(x[2 * p], x[2 * p + 1]));
    }
    if (__builtin_expect(nan != 0, 0)) {
        // A NaN becomes the canonical 0x7FFF (as round_pair_bf16).
#pragma unroll
        for (int p = 0; p < kHalfSteps / 2; ++p) {
            if (__builtin_isnan(x[2 * p])) h.r[p] = (h.r[p] & 0xFFFF0000u) | 0x7FFFu;
            if (__builtin_isnan(x[2 * p + 1])) h.r[p] = (h.r[p] & 0xFFFFu) | 0x7FFF0000u;
        }
    }
    if (!kFull) {
#pragma unroll
        for (int p = 0; p < kHalfSteps / 2; ++p) {
            const uint32_t off0 = half_offset(first, mask, 2 * p);
            if (off0 >= valid) h.r[p] = 0u;   // so is the row after it
            else if (off0 + kLanes >= valid) h.r[p] &= 0xFFFFu;
        }
    }
}

// The half's side bytes into rows 0..7 of `rows` (64 bytes each).
__device__ __forceinline__ void store_half_sides(const HalfEmit &h, uint8_t *rows) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int p = 0; p < kHalfSteps / 2; ++p) {
        // The mantissa and, from r >> 8, the sign of each half.
        const uint32_t r = h.r[p], sign_down = r >> 8;
        uint32_t side0, side1;
        asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(side0) : "s"(0x7Fu), "v"(r), "v"(sign_down));
        asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(side1) : "s"(0x007F0000u), "v"(r), "v"(sign_down));
        rows[2 * p * kWave + lane] = static_cast<uint8_t>(side0);
        rows[(2 * p + 1) * kWave + lane] = static_cast<uint8_t>(side1 >> 16);
    }
}

// The encode entries of quad `q` (0 or 1) of the half.
template <bool kFull>
__device__ __forceinline__ void look_up_quad(HalfEmit &h, const uint2 *enc, int q, int first,
                                             uint32_t mask, uint32_t valid) {
#pragma unroll
    for (int p = 2 * q; p < 2 * q + 2; ++p) {
        const uint32_t x = exponent_bytes(h.r[p]);
        h.e[2 * p] = enc[x & 255u];
        h.e[2 * p + 1] = enc[(x >> 16) & 255u];
        if (!kFull) {
            // Positions past the logical end carry no code (encode.py:255-256).
            const uint32_t off0 = half_offset(first, mask, 2 * p);
            if (off0 >= valid) h.e[2 * p] = make_uint2(0u, 0u);
            if (off0 + kLanes >= valid) h.e[2 * p + 1] = make_uint2(0u, 0u);
        }
    }
}

// The codes of the half's quad `q` as two pairs' bits.
struct QuadCodes {
    uint32_t code0, code1, len0, len1;

    __device__ __forceinline__ QuadCodes(const HalfEmit &h, int q) {
        const uint2 *e = h.e + 4 * q;
        code0 = e[0].x | (e[1].x << e[0].y);
        code1 = e[2].x | (e[3].x << e[2].y);
        len0 = e[0].y + e[1].y;
        len1 = e[2].y + e[3].y;
    }
};

// Append both quads' codes, which are known to fit: a quad in one piece unless
// some lane's codes are more than 32 bits (each pair is at most 32).
__device__ __forceinline__ void put_half(const QuadCodes &a, const QuadCodes &b,
                                         StreamWriter &writer) {
    const uint32_t len_a = a.len0 + a.len1, len_b = b.len0 + b.len1;
    if (__builtin_expect(__any(max(len_a, len_b) > 32u), 0)) {
        writer.put_bits(a.code0, a.len0);
        writer.put_bits(a.code1, a.len1);
        writer.put_bits(b.code0, b.len0);
        writer.put_bits(b.code1, b.len1);
    } else {
        writer.put_bits(a.code0 | (a.code1 << (a.len0 & 31u)), len_a);
        writer.put_bits(b.code0 | (b.code1 << (b.len0 & 31u)), len_b);
    }
    writer.fits += kHalfSteps / 2;
}

// Near a stream's end, pair by pair, with the exponent bytes of an overflowing
// pair's rows going to the exponent array (positions past the tensor's end are
// outside its resource and are dropped).
__device__ __forceinline__ void put_half_by_pairs(const HalfEmit &h, StreamWriter &writer,
                                                  int first, uint32_t mask,
                                                  __amdgpu_buffer_rsrc_t exponents) {
#pragma unroll
    for (int p = 0; p < kHalfSteps / 2; ++p) {
        const bool over = writer.put(h.e[2 * p], h.e[2 * p + 1]);
        const uint32_t off = over ? half_offset(first, mask, 2 * p) : kOutOfRange;
        uint32_t r = h.r[p];
        asm("" : "+v"(r));   // shifted here, on the rare path only
        __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(r >> 7), exponents, off, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(r >> 23), exponents,
                                             off + kLanes, 0, 0);
    }
}

}  // namespace lct
