// Device functions of the kernels that multiply float32 values as three bfloat16 pieces each: piece
// matrices in memory, their tiles in LDS, and the copies from one to the other.
//
// Piece matrix: row r, column k, piece q at  r * pitch + (k / 32) * 192 + q * 64 + (k % 32) * 2  bytes:
// the three pieces of 32 columns lie together, and a slab of a row is 192 consecutive bytes.  Columns
// are filled with zeros to a multiple of 32.
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

// neighbouring lanes' values (lane ^ 1)
DEVINL float swap1(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));
}
DEVINL float swap2(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));
}

// four columns of a piece-matrix row, k % 4 == 0.  (An infinity's pieces are infinity, NaN, NaN: the first
// alone is the value.)
DEVINL float4 load_pieces4(const char* row, int k) {
    const char* p = row + (size_t)(k >> 5) * 192 + (k & 31) * 2;
    const uint2 hi = *reinterpret_cast<const uint2*>(p);
    float4 v = make_float4(bf16_lo_f32(hi.x), bf16_hi_f32(hi.x), bf16_lo_f32(hi.y), bf16_hi_f32(hi.y));
    const float4 first = v;
#pragma unroll
    for (int q = 1; q < 3; ++q) {
        const uint2 raw = *reinterpret_cast<const uint2*>(p + 64 * q);
        v.x += bf16_lo_f32(raw.x); v.y += bf16_hi_f32(raw.x);
        v.z += bf16_lo_f32(raw.y); v.w += bf16_hi_f32(raw.y);
    }
    if (!(fabsf(first.x) < INFINITY)) v.x = first.x;
    if (!(fabsf(first.y) < INFINITY)) v.y = first.y;
    if (!(fabsf(first.z) < INFINITY)) v.z = first.z;
    if (!(fabsf(first.w) < INFINITY)) v.w = first.w;
    return v;
}
DEVINL float load_piece1(const char* row, int k) {
    const char* p = row + (size_t)(k >> 5) * 192 + (k & 31) * 2;
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < 3; ++q) v += bf16_to_f32(*reinterpret_cast<const uint16_t*>(p + 64 * q));
    return v;
}
DEVINL void store_pieces4(char* row, int k, float4 v) {
    uint2 piece[3];
    split4_bf16(as_x4(v), piece);
    char* p = row + (size_t)(k >> 5) * 192 + (k & 31) * 2;
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(p + 64 * q) = piece[q];
}
// two neighbouring values -> three words of two pieces each
DEVINL void split2(float a, float b, uint32_t w[3]) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        w[q] = pack_bf16(a, b);
        if (q < 2) { a -= bf16_lo_f32(w[q]); b -= bf16_hi_f32(w[q]); }
    }
}

// --------------------------------------------------------------------------
// tiles in LDS

// Contraction-innermost operand: R rows x 32 columns of a piece matrix as [piece][row][32], a row's
// four 16-byte chunks at position chunk ^ ((row / 4) % 4): sixteen rows' reads of one chunk fall on
// all banks.  One copy instruction moves sixteen rows of one piece.
template <int R>
struct RowTile {
    static constexpr int kBytes = 3 * R * 64, kCopies = 3 * R / 16;
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
template <int C>
struct ColTile {
    static constexpr int kBytes = 3 * 32 * C * 2, kCopies = 3 * C / 16;
    static constexpr int kKey = C >= 128 ? 3 : 1;  // (a row of 64 columns has four units)
    // (rows past `last` repeat it)
    static DEVINL uint32_t source(int x, int lane, int pitch, int last = 31) {
        constexpr int chunks = C / 8, rows = 64 / chunks;
        const int piece = x / (C / 16), row = (x % (C / 16)) * rows + lane / chunks, pos = lane % chunks;
        const int chunk = pos ^ ((row & kKey) << 2);  // 16-byte chunks: two to a unit
        const int col = chunk * 8;
        return (uint32_t)(min(row, last) * pitch + (col >> 5) * 192 + piece * 64 + (col & 31) * 2);
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
