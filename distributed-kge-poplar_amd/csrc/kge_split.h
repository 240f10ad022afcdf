// Device functions of the kernels that multiply float32 values as pieces of 16 bits: piece matrices in
// memory, their tiles in LDS, and the copies from one to the other.  A value is three bfloat16 pieces, or
// two float16 halves (below).
//
// Piece matrix of NP pieces: row r, column k, piece q at  r * pitch + (k / 32) * 64 NP + q * 64 + (k % 32) * 2
// bytes: the pieces of 32 columns lie together, and a slab of a row is 64 NP consecutive bytes.
// Columns are filled with zeros to a multiple of 32.
#pragma once

#include "kge_device.h"

namespace kge {

// --------------------------------------------------------------------------
// global memory -> LDS copies and their waits

// 64 lanes x 16 bytes: lane l's bytes at base + off go to LDS byte lds + 16 l (base, lds: wave-uniform)
DEVINL void lds_copy16(const char* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
// until at most N of this wave's memory operations are under way, then for the workgroup's other waves
template <int N>
DEVINL void wait_copies_and_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
DEVINL uint32_t lds_address(const void* p) {
    return (uint32_t)(size_t)(const __attribute__((address_space(3))) char*)p;
}

// neighbouring lanes' values (lane ^ 1, lane ^ 2); the lane's mirror image in its half row of eight, in its row of 16
template <int CTRL>
DEVINL float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
DEVINL float mirror8(float v) { return dpp<0x141>(v); }
DEVINL float mirror16(float v) { return dpp<0x140>(v); }
DEVINL float swap1(float v) {
    return dpp<0xB1>(v);
}
DEVINL float swap2(float v) {
    return dpp<0x4E>(v);
}

DEVINL void store_pieces4(char* row, int k, float4 v) {
    uint2 piece[3];
    split4_bf16(as_x4(v), piece);
    char* p = row + (size_t)(k >> 5) * 192 + (k & 31) * 2;
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(p + 64 * q) = piece[q];
}

// --------------------------------------------------------------------------
// Float16 halves.  x = s (h0 + h1 / 2048), h0 = float16(x / s), h1 = float16(2048 (x / s - h0)): 11 bits
// each, the rounding of h0 to either side worth one more, so the sum differs from x by at most one unit in its
// 24th bit, and for three values of four by nothing.  The scale s is a power of two that brings the largest of a
// row (or of a block of coefficients) to 2^14; with the second half 2^11 times as large as it counts, both are
// normal float16 numbers down to 2^-28 of that largest value, and what is smaller is off by 2^-49 of it at most.  Where a
// column is that small in one row after the other, and so in every gradient, they are wide ones: their places hold them as
// float32, their scales are NaN, and their pairs and sub-blocks are taken in the direct forms.
//   a b = sa sb (a0 b0 + (a0 b1 + a1 b0) / 2048 + O(2^-24 |a0 b0|)):
// three matrix instructions where three bfloat16 pieces take six, two fragments of an operand where they take
// three, and a row of halves is as long as the float32 row.  The cross products have an accumulator of their own.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
constexpr float kHalfStep = 1.f / 2048.f;
constexpr int kHalfBytes = 128;  // of 32 columns of a row

// the scale for a largest magnitude (not negative; infinities and NaN take some scale, their halves say the rest).
// Rows below 2^-112 share one: it and its reciprocal are normal numbers.  Rows of zeros, which any scale would do for, have
// an ordinary row's: their coefficients carry it and stand beside the other rows' in one block.
DEVINL float half_scale(float largest) {
    const int e = largest == 0.f ? 0 : min(max((int)(__float_as_uint(largest) >> 23) - 127, -112), 127);
    return __uint_as_float((uint32_t)(e - 14 + 127) << 23);
}
// a power of two's exponent, its reciprocal
DEVINL int pow2_exponent(float s) { return (int)(__float_as_uint(s) >> 23) - 127; }
DEVINL float pow2_inverse(float s) { return __uint_as_float(0x7f000000u - __float_as_uint(s)); }
// The scale of a wide row, among the exponents of scales, and where its columns k .. k + 3 (k % 4 == 0) lie: eight columns are
// the sixteen bytes of their first halves and then those of the second ones.
constexpr float kLeastHalf = 0x1p-14f;
constexpr int kWideExponent = 128;
DEVINL float wide_scale() { return __uint_as_float(0x7fc00000u); }
DEVINL bool is_wide(float scale) { return scale != scale; }
DEVINL size_t wide_at(int k) { return (size_t)(k >> 5) * kHalfBytes + (k & 4) * 16 + ((k & 31) >> 3) * 16; }
// Coefficients are halves with a scale per block, whose largest comes to 2^11 .. 2^15; those below kSmallCoef can go to a
// matrix of their own, 2^kSmallShift times as large.
constexpr float kSmallCoef = 0x1p-13f;
constexpr int kSmallShift = 28;
// two values, scaled already -> two words of two halves each
DEVINL void split2_f16(float a, float b, uint32_t w[2]) {
    const f16x2 h = {(_Float16)a, (_Float16)b};
    const f16x2 l = {(_Float16)((a - (float)h.x) * 2048.f), (_Float16)((b - (float)h.y) * 2048.f)};
    w[0] = __builtin_bit_cast(uint32_t, h);
    w[1] = __builtin_bit_cast(uint32_t, l);
}
// Four columns of a row of halves, k % 4 == 0.  The second halves are cut off here, not rounded, and what that leaves
// is one bit: whether the value has a twelfth bit there.  A whole wave at once; lost[i]: bit l for lane l's column k + i.
DEVINL void store_halves4(char* row, int k, float4 v, bool live, uint64_t (&lost)[4]) {
    const float x[4] = {v.x, v.y, v.z, v.w};
    uint32_t w[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const f16x2 h = {(_Float16)x[2 * i], (_Float16)x[2 * i + 1]};
        const float a = (x[2 * i] - (float)h.x) * 2048.f, b = (x[2 * i + 1] - (float)h.y) * 2048.f;
        const auto cut = __builtin_amdgcn_cvt_pkrtz(a, b);
        const f16x2 l = __builtin_bit_cast(f16x2, cut);
        lost[2 * i] = __ballot(a != (float)l.x);
        lost[2 * i + 1] = __ballot(b != (float)l.y);
        w[0][i] = __builtin_bit_cast(uint32_t, h);
        w[1][i] = __builtin_bit_cast(uint32_t, l);
    }
    if (!live) return;
    char* p = row + (size_t)(k >> 5) * kHalfBytes + (k & 31) * 2;
#pragma unroll
    for (int q = 0; q < 2; ++q) *reinterpret_cast<uint2*>(p + 64 * q) = make_uint2(w[q][0], w[q][1]);
}
// The rows of a gather as they were.
DEVINL float join_lost(_Float16 h, _Float16 l, uint32_t bit) {  // (of a finite value, without its scale)
    return fmaf(__uint_as_float(__float_as_uint((float)l) + (bit << 12)), kHalfStep, (float)h);
}
DEVINL float with_lost(_Float16 h, _Float16 l, bool lost, float scale) {
    if (!(fabsf((float)h) < INFINITY)) return (float)h;
    return join_lost(h, l, lost) * scale;
}
// eight columns k .. k + 7 of row c (k % 8 == 0), all loads in one go
struct Row8 {
    uint4 h, l;
    uint32_t lost;
    float scale;
    DEVINL void load(const SplitRows& s, int c, int k) {
        const char* p = s.halves + (size_t)c * half_pitch(s.Kp) + (size_t)(k >> 5) * kHalfBytes + (k & 31) * 2;
        h = *reinterpret_cast<const uint4*>(p);
        l = *reinterpret_cast<const uint4*>(p + 64);
        lost = s.lost[(size_t)c * (s.Kp >> 5) + (k >> 5)] >> ((k & 31) >> 2);
        scale = s.scale[c];
    }
    template <int I, bool WIDE>  // (WIDE: it may be a wide row)
    DEVINL float value() const {
        constexpr int W = I >> 1;
        if (WIDE && is_wide(scale)) {
            const uint4 four = I < 4 ? h : l;
            return __uint_as_float((I & 3) == 0 ? four.x : (I & 3) == 1 ? four.y : (I & 3) == 2 ? four.z : four.w);
        }
        const f16x2 hw = __builtin_bit_cast(f16x2, W == 0 ? h.x : W == 1 ? h.y : W == 2 ? h.z : h.w);
        const f16x2 lw = __builtin_bit_cast(f16x2, W == 0 ? l.x : W == 1 ? l.y : W == 2 ? l.z : l.w);
        return with_lost(I & 1 ? hw.y : hw.x, I & 1 ? lw.y : lw.x, (lost >> lost_at(I)) & 1u, scale);
    }
};
struct Row1 {  // one column of a row whose scale is known
    uint32_t h, l, lost;
    DEVINL void load(const SplitRows& s, int c, int k, float scale) {
        const char* const row = s.halves + (size_t)c * half_pitch(s.Kp);
        const uint32_t at = is_wide(scale) ? (uint32_t)wide_at(k) + (k & 3) * 4 : (uint32_t)((k >> 5) * kHalfBytes + (k & 31) * 2);
        h = *reinterpret_cast<const uint16_t*>(row + at);
        l = *reinterpret_cast<const uint16_t*>(row + at + (is_wide(scale) ? 2 : 64));  // (a wide row's: the upper half of the value)
        lost = s.lost[(size_t)c * (s.Kp >> 5) + (k >> 5)];
    }
    DEVINL float value(int k, float scale) const {
        if (is_wide(scale)) return __uint_as_float(h | l << 16);
        return with_lost(__builtin_bit_cast(_Float16, (uint16_t)h), __builtin_bit_cast(_Float16, (uint16_t)l), (lost >> lost_at(k)) & 1u, scale);
    }
};

// --------------------------------------------------------------------------
// tiles in LDS

// Contraction-innermost operand: R rows x 32 columns of a piece matrix as [piece][row][32], a row's
// four 16-byte chunks at position chunk ^ ((row / 4) % 4): sixteen rows' reads of one chunk fall on
// all banks.  One copy instruction moves sixteen rows of one piece.
template <int R, int NP = 3>
struct RowTile {
    static constexpr int kBytes = NP * R * 64, kCopies = NP * R / 16;
    // offset of copy x's bytes for this lane, from the tile's first row and slab
    static DEVINL uint32_t source(int x, int lane, int pitch) {
        const int piece = x / (R / 16), row = (x % (R / 16)) * 16 + (lane >> 2);
        const int chunk = (lane & 3) ^ ((row >> 2) & 3);
        return (uint32_t)(row * pitch + piece * 64 + chunk * 16);
    }
    // the 16-column step `ks`'s fragment of rows row0 .. row0 + 31 (this lane: row row0 + lane % 32)
    static DEVINL floatx4 fragment(const char* tile, int piece, int row0, int ks, int lane) {
        const int row = row0 + (lane & 31), chunk = (2 * ks + (lane >> 5)) ^ ((row >> 2) & 3);
        return *reinterpret_cast<const floatx4*>(tile + piece * (R * 64) + row * 64 + chunk * 16);
    }
};

// Contraction-outermost operand: 32 rows (contraction) x C columns of a piece matrix as
// [piece][row][C], read back transposed (ds_read_b64_tr_b16: sixteen lanes read a 4 x 16 block and
// each receives one column of it).  A row's 32-byte units sit at position unit ^ 2 (row % 4): the four
// rows that a read instruction's half takes fall on different banks.  One copy instruction moves
// 512 / C rows of one piece.
template <int C, int NP = 3>
struct ColTile {
    static constexpr int kBytes = NP * 32 * C * 2, kCopies = NP * C / 16;
    static constexpr int kKey = C >= 128 ? 3 : 1;  // (a row of 64 columns has four units)
    // (rows past `last` repeat it)
    static DEVINL uint32_t source(int x, int lane, int pitch, int last = 31) {
        constexpr int chunks = C / 8, rows = 64 / chunks;
        const int piece = x / (C / 16), row = (x % (C / 16)) * rows + lane / chunks, pos = lane % chunks;
        const int chunk = pos ^ ((row & kKey) << 2);  // 16-byte chunks: two to a unit
        const int col = chunk * 8;
        return (uint32_t)(min(row, last) * pitch + (col >> 5) * (64 * NP) + piece * 64 + (col & 31) * 2);
    }
    // columns col0 .. col0 + 31 over the sixteen rows of step `ks` (this lane: column
    // col0 + lane % 32, rows 8 (lane / 32) .. + 7)
    static DEVINL floatx4 fragment(const char* tile, int piece, int col0, int ks, int lane) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        typedef const __attribute__((address_space(3))) s16x4* lds_ptr;
        const int g = lane >> 4, r4 = (lane & 15) >> 2;
        const int unit = ((col0 >> 4) + (g & 1)) ^ ((r4 & kKey) << 1);
        const char* p = tile + piece * (64 * C) + (16 * ks + 8 * (g >> 1) + r4) * (2 * C) + unit * 32 + (lane & 3) * 8;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(lds_ptr)p);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(lds_ptr)(p + 4 * 2 * C));
        typedef short s16x8 __attribute__((ext_vector_type(8)));
        return __builtin_bit_cast(floatx4, s16x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
    }
};

}  // namespace kge
