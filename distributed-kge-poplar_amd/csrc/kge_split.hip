// gfx950 scoring kernels on float16 halves (L2 and dot): the operand gather, the forward scores with the
// fused loss, and both sides of the backward.
//
// A float32 value is a scale and two float16 halves, and a float32 product is three products of halves
// (kge_split.h).  Every value is split once, by the kernel that makes it: the gather writes the
// operand rows as halves, the forward writes the backward's coefficients as halves, and the product
// kernels copy tiles straight from memory into LDS (global_load_lds, no registers, no vector
// instructions), so that their waves do little else than read fragments and multiply.
//
#include "kge_device.h"
#include "kge_loss.h"
#include "kge_split.h"

#include <algorithm>
#include <cstdint>

namespace kge {

// --------------------------------------------------------------------------
// reductions over a wave without a way through LDS: the result is in lane 63 (rows of 16 by DPP, then across them)
template <class Op>
DEVINL float wave_reduce63(float v, Op&& op) {
    v = op(v, swap1(v));
    v = op(v, swap2(v));
    v = op(v, mirror8(v));
    v = op(v, mirror16(v));
    const int x = __float_as_int(v);
    v = op(v, __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0x142, 0xa, 0xf, false)));  // row 0's to 1, 2's to 3
    const int y = __float_as_int(v);
    return op(v, __int_as_float(__builtin_amdgcn_update_dpp(y, y, 0x143, 0xc, 0xf, false)));  // 1's to 2 and 3
}
// the largest of a wave's magnitudes, as its bits
DEVINL uint32_t wave_max_bits(float v) {
    v = wave_reduce63(v, [](float a, float b) { return fmaxf(a, b); });
    return (uint32_t)__builtin_amdgcn_readlane(__float_as_int(v), 63);
}

// --------------------------------------------------------------------------
// operand gather: RPW contributions per wave, their entity (or hidden) rows with the relation
// applied for the heads, as halves; and the rows' scales and squared norms.  Workgroup (d, y, z): a lot of
// block d's B heads and then T tails (z: a grid's y ends at 65535).  Where S is a multiple of 8, that runs on the XCD (d % 8) of the
// block's tiles.
// ET: the rows' element type, or -1: as `ent` says, the complex product and the rotation among the
// relations; ONE: rows of at most 256 columns, which stay in their registers between the largest value and the halves.
template <int RPW, int ET, bool ONE>
__global__ __launch_bounds__(256, 8) void k_gather_halves(RowSource ent, const float* __restrict__ rel, const uint32_t* __restrict__ crel,
                                                       int rel_mode, int half, SplitRows s, const uint32_t* __restrict__ tcount,
                                                       int B, int T, int tpad) {
    constexpr bool XF = ET < 0;
    const int lane = threadIdx.x & 63, d = blockIdx.x;
    const int i0 = ((blockIdx.z * gridDim.y + blockIdx.y) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * RPW;
    // the row numbers are asked for together with the block's tail count (rows past it are
    // never used, but their slots hold valid numbers): one round trip instead of two.  (All of them
    // are the wave's, and scalar loads: a lane has an offset into its rows and no addresses.)
    int c[RPW];
    uint32_t key[RPW], rkey[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        const int i = min(i0 + r, B + T - 1);  // a row past the end repeats the last one
        c[r] = i < B ? d * B + i : s.n_head + d * T + i - B;
        key[r] = ent.index ? ent.index[c[r]] : (uint32_t)c[r];
        rkey[r] = (i < B && rel_mode) ? crel[c[r]] : 0u;
    }
    // (rows behind a block's distinct tails repeat its first one, and what they hold meets coefficients of zero: halves, always)
    const int end = B + tail_limit(tcount, d, T, tpad), live = B + (tcount ? (int)tcount[d] : T);
#pragma unroll
    for (int r = 0; r < RPW; ++r) asm volatile("" : "+s"(key[r]), "+s"(rkey[r]));
    if (i0 >= end) return;
    const char* row[RPW];
    const float* rrow[RPW];
    float sq[RPW], top[RPW], least[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        row[r] = ent.base + (int64_t)key[r] * ent.pitch;
        rrow[r] = (i0 + r < B && rel_mode) ? rel + (size_t)rkey[r] * s.Dp : nullptr;
        sq[r] = top[r] = 0.f;
        least[r] = INFINITY;
    }
    float4 v[RPW];
    auto fetch = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < RPW; ++r) v[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (k >= s.Dp) return;
#pragma unroll
        for (int r = 0; r < RPW; ++r) v[r] = XF ? load4(row[r], k, ent) : load4(row[r], k, ET);  // all loads first
        float4 w[RPW];
#pragma unroll
        for (int r = 0; r < RPW; ++r)
            if (rrow[r] && !(XF && rel_mode >= 3)) w[r] = *reinterpret_cast<const float4*>(rrow[r] + k);
#pragma unroll
        for (int r = 0; r < RPW; ++r)
            if (rrow[r]) {
                if (XF && rel_mode >= 3) v[r] = relation_xf(v[r], row[r], ent.etype, rrow[r], k, half, rel_mode);
                else v[r] = rel_mode == 1 ? f4add(v[r], w[r]) : f4mul(v[r], w[r]);
            }
    };
    const int k_end = ONE ? 256 : (s.Kp + 255) & ~255;  // (the whole wave stays together)
    for (int k = lane * 4; k < k_end; k += 256) {
        fetch(k);
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            sq[r] += v[r].x * v[r].x + v[r].y * v[r].y + v[r].z * v[r].z + v[r].w * v[r].w;
            top[r] = fmaxf(fmaxf(top[r], fmaxf(fabsf(v[r].x), fabsf(v[r].y))), fmaxf(fabsf(v[r].z), fabsf(v[r].w)));
            if (k < s.Dp) least[r] = fminf(fminf(least[r], fminf(fabsf(v[r].x), fabsf(v[r].y))), fminf(fabsf(v[r].z), fabsf(v[r].w)));
        }
    }
    // Seldom (or where there are zeros): whether some element of row i is too small for halves, and not zero, and the next
    // three rows' of its column are too.  Of ordinary rows' elements one in 10^8 is so small by chance, and then the others make up its
    // column of every gradient.  (With a row in the direct form for each of those, a step of 64 blocks of 256 x 512 took 2 us
    // more on average, one of 16 blocks of 256 x 1536 7.)
    auto small_column = [&](int i) __attribute__((always_inline)) {
        const int first = i < B ? 0 : B, n = i < B ? B : live - B;
        auto row4 = [&](int x, int k) __attribute__((always_inline)) {
            if (k >= s.Dp) return make_float4(0.f, 0.f, 0.f, 0.f);
            const int at = first + (i - first + x) % n, c = at < B ? d * B + at : s.n_head + d * T + at - B;
            const char* const row = ent.base + (int64_t)(ent.index ? ent.index[c] : (uint32_t)c) * ent.pitch;
            const float4 v = XF ? load4(row, k, ent) : load4(row, k, ET);
            if (at >= B || !rel_mode) return v;
            const float* const rrow = rel + (size_t)crel[c] * s.Dp;
            if (XF && rel_mode >= 3) return relation_xf(v, row, ent.etype, rrow, k, half, rel_mode);
            const float4 w = *reinterpret_cast<const float4*>(rrow + k);
            return rel_mode == 1 ? f4add(v, w) : f4mul(v, w);
        };
#pragma unroll 1
        for (int k0 = 0; k0 < k_end; k0 += 256) {  // for each of the rows its largest element, then the lane's four of these columns
            int is = 15;
            float limit = 0.f;
#pragma unroll 1
            for (int t = 0; t < 8 && __ballot(is); ++t) {
                const bool look = t & 1;
                float most = 0.f;
#pragma unroll 1
                for (int q = look ? k0 : 0; q < (look ? k0 + 1 : k_end); q += 256) {
                    const float4 a = row4(t >> 1, q + 4 * lane);
                    most = fmaxf(fmaxf(most, fmaxf(fabsf(a.x), fabsf(a.y))), fmaxf(fabsf(a.z), fabsf(a.w)));
                    if (!look) continue;
                    is &= (fabsf(a.x) < limit) | (fabsf(a.y) < limit) << 1 | (fabsf(a.z) < limit) << 2 | (fabsf(a.w) < limit) << 3;
                    if (t == 1) is &= (a.x != 0.f) | (a.y != 0.f) << 1 | (a.z != 0.f) << 2 | (a.w != 0.f) << 3;
                }
                if (!look) limit = kLeastHalf * half_scale(__uint_as_float(wave_max_bits(most)));
            }
            if (__ballot(is)) return true;
        }
        return false;
    };
    float up[RPW], sum[RPW];
    uint32_t look = 0u, wide = 0u;  // rows' bits
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        sum[r] = wave_reduce63(sq[r], [](float a, float b) { return a + b; });
        const float most = __uint_as_float(wave_max_bits(top[r]));
        up[r] = pow2_inverse(half_scale(most));
        if (__ballot(least[r] * up[r] < kLeastHalf) && most < INFINITY && i0 + r < live) look |= 1u << r;
    }
    if (__builtin_expect(look != 0u, 0)) {
#pragma unroll 1
        for (; look; look &= look - 1u)
            if (small_column(i0 + __ffs((int)look) - 1)) wide |= look & (0u - look);
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): without it, the waits for these loads come behind the stores below, and for those
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r)
        if (lane == 63 && i0 + r < end) {
            s.norm[c[r]] = sum[r];
            s.scale[c[r]] = (wide >> r) & 1u ? wide_scale() : pow2_inverse(up[r]);
        }
    for (int k = lane * 4; k < k_end; k += 256) {
        if (!ONE) fetch(k);
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            if (__builtin_expect((wide >> r) & 1u, 0)) {
                if (i0 + r < end && k < s.Kp)
                    *reinterpret_cast<float4*>(s.halves + (size_t)c[r] * half_pitch(s.Kp) + wide_at(k)) = v[r];
                continue;
            }
            uint64_t lost[4];
            store_halves4(s.halves + (size_t)c[r] * half_pitch(s.Kp), k,
                          make_float4(v[r].x * up[r], v[r].y * up[r], v[r].z * up[r], v[r].w * up[r]), i0 + r < end && k < s.Kp, lost);
            // a slab's 32 bits: a byte of each ballot, by one lane
            uint32_t word = 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i) word |= (((uint32_t)(lane & 4 ? lost[i] >> 32 : lost[i]) >> (8 * (lane & 3))) & 255u) << (8 * i);
            const int slab = ((k - 4 * lane) >> 5) + lane;
            if (lane < 8 && slab < s.Kp >> 5 && i0 + r < end) s.lost[(size_t)c[r] * (s.Kp >> 5) + slab] = word;
        }
    }
}

void launch_gather_halves(const RowSource& ent, const float* rel, const uint32_t* crel, int rel_mode, int half,
                          const SplitRows& s, const ScoreShape& sh, hipStream_t stream) {
    // two rows per wave where that leaves enough waves: the kernel is resident waves over the
    // latency of the chain row number -> row -> store, and a wave may as well keep two chains going
    auto grid = [&](int rows) {
        const unsigned lots = (unsigned)((sh.B + sh.T + rows - 1) / rows), y = std::min(lots, 32768u);
        return dim3((unsigned)sh.S, y, (lots + y - 1) / y);
    };
#define KGE_GATHER(N_, ET_, ONE_)                                                                                       \
    hipLaunchKernelGGL((k_gather_halves<N_, ET_, ONE_>), grid(4 * N_), dim3(256), 0, stream, \
                       ent, rel, crel, rel_mode, half, s, sh.tcount, sh.B, sh.T, sh.tpad)
#define KGE_GATHER_ET(ET_)                                                                                      \
    do {                                                                                                        \
        if (s.Kp > 256) KGE_GATHER(1, ET_, false);                                                              \
        else if (s.n_rows >= 8192) KGE_GATHER(2, ET_, true);                                                    \
        else KGE_GATHER(1, ET_, true);                                                                          \
    } while (0)
    if (rel_mode >= 3 || !ent.vec) { if (s.Kp > 256) KGE_GATHER(1, -1, false); else KGE_GATHER(1, -1, true); }
    else if (ent.etype == ET_F32) KGE_GATHER_ET(ET_F32);
    else if (ent.etype == ET_BF16) KGE_GATHER_ET(ET_BF16);
    else KGE_GATHER_ET(ET_F16);
#undef KGE_GATHER_ET
#undef KGE_GATHER
}

// --------------------------------------------------------------------------
// products

// Tiles of TM x TN, waves as WM x WN of them, 32 x 32 of the tile to a wave: EU waves to a SIMD, whose registers allow as many
// workgroups as LDS has room for (three of 128 x 64, four of 64 x 64).  What a launch spends its time on is the first slab's
// way from memory, the loop and the epilogue of every workgroup, one after the other; workgroups beside it fill
// the gaps, and a third of 128 x 64 is worth more than a third tile copy (64 blocks of 256 x 512, 331 distinct tails, D = 256:
// forward 35.5 us with two workgroups of three copies, 30.2 with three of two; backward 49.9 and 43.8).
template <int TM_, int TN_, int WM_, int WN_, int EU_>
struct SplitTile { static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, EU = EU_, threads = WM_ * WN_ * 64; };
using TileSmall = SplitTile<64, 64, 2, 2, 4>;
using TileLarge = SplitTile<128, 64, 4, 2, 6>;

// The product loop of a tile: n_slab slabs of 32 contraction steps, two tile copies in LDS
// (one fills while the other is multiplied, one barrier per slab).  TA, TB: RowTile / ColTile;
// a_step, b_step: bytes from slab to slab.  Each wave's 32 x 32 of the tile in two accumulators:
// `big` the products of first halves, `small` the cross products.
// b_rows: rows of `b` along the contraction where it lies across it (ColTile).  The last slab's rows past them
// repeat the last one: their coefficients are zero, but what lies behind a block's rows are other
// blocks', and zero times a neighbour's infinity or NaN would be this block's NaN.
template <class TA, class TB, class Tile>
struct SplitProduct {
    static constexpr int NW = Tile::WM * Tile::WN, kCopy = TA::kBytes + TB::kBytes, kLds = 2 * kCopy;
    static_assert(Tile::TM == 32 * Tile::WM && Tile::TN == 32 * Tile::WN, "one 32 x 32 block to a wave");
    static constexpr int kCopies = TA::kCopies + TB::kCopies, kEach = kCopies / NW;
    static_assert(kCopies % NW == 0, "every wave issues the same number of copies");

    // meanwhile(): what the caller has to fetch for itself, under the first slab's way from memory;
    // before(slab): ahead of the slab's products, whether to form them
    template <class Meanwhile, class Before>
    static DEVINL void run(char* smem, const char* a, int a_pitch, size_t a_step, const char* b, int b_pitch, size_t b_step,
                           int n_slab, int b_rows, floatx16& big, floatx16& small, int lane, int wave,
                           Meanwhile&& meanwhile, Before&& before) {
        uint32_t off[kEach];
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
            const int x = wave + NW * i;
            off[i] = x < TA::kCopies ? TA::source(x, lane, a_pitch) : TB::source(x - TA::kCopies, lane, b_pitch);
        }
        const uint32_t lds0 = lds_address(smem);
        auto fill = [&](int slab) __attribute__((always_inline)) {
            const char* as = a + slab * a_step;
            const char* bs = b + slab * b_step;
            const uint32_t to = lds0 + (slab & 1) * kCopy;
            if constexpr (!std::is_same_v<TB, RowTile<Tile::TN, 2>>) {
                const int last = b_rows - 32 * slab - 1;
                if (last < 31)  // the last slab's offsets take the others' place
#pragma unroll
                    for (int i = 0; i < kEach; ++i) {
                        const int x = wave + NW * i;
                        if (x >= TA::kCopies) off[i] = TB::source(x - TA::kCopies, (int)lane_here(), b_pitch, last);
                    }
            }
#pragma unroll
            for (int i = 0; i < kEach; ++i) {
                const int x = wave + NW * i;
                lds_copy16(x < TA::kCopies ? as : bs, off[i], to + x * 1024);
            }
        };
        fill(0);
        meanwhile();
#pragma unroll
        for (int r = 0; r < 16; ++r) big[r] = small[r] = 0.f;
        const int wm = 32 * (wave / Tile::WN), wn = 32 * (wave % Tile::WN);
        for (int slab = 0; slab < n_slab; ++slab) {
            wait_copies_and_barrier<0>();
            const bool count = before(slab);  // (ahead of the copies: behind them, its wait for
            // exponents that it may have loaded was one for the next slab, 55 -> 44 us of 16 blocks of 256 x 1536)
            if (slab + 1 < n_slab) fill(slab + 1);
            if (!count) continue;
            const char* ta = smem + (slab & 1) * kCopy;
            const char* tb = ta + TA::kBytes;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                floatx4 fa[2], fb[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    fa[q] = TA::fragment(ta, q, wm, ks, lane);
                    fb[q] = TB::fragment(tb, q, wn, ks, lane);
                }
                auto product = [&](int qa, int qb, floatx16& acc) __attribute__((always_inline)) {
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fa[qa]), __builtin_bit_cast(f16x8, fb[qb]), acc, 0, 0, 0);
                };
                product(0, 0, big);
                product(0, 1, small);
                product(1, 0, small);
            }
        }
    }
};

// --------------------------------------------------------------------------
// the coefficient matrix as halves

// A 32 x 32 block of coefficients lies in accumulator layout: register r of lane l is row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.  The backward multiplies rows of halves that lack their scales, the
// heads' on one side and the tails' on the other: a coefficient takes both along, and the backward takes its own
// row's out of the finished sum.  The block's own scale is 2^exponent, a multiple of four, so that the backward seldom
// meets another one in the next block; its largest comes to 2^11 at least.  Halves hold 22 bits down to 2^-14, and what a
// row's or a column's gradient is made of is its own largest: where one's lies below 2^-13 (an odd row out, a tail that no
// head's softmax gives a probability worth mentioning), the coefficients below that go to a matrix of their own, 2^28 times
// as large.  Where even that is not enough, the block is taken in the direct form.

// sums (or maxima) of a block's rows: at each step a lane keeps half of its rows and hands the other half's over.  The
// result's row is the one that register lane % 16 holds, in all lanes of that row's half.
template <class Value, class Op>
DEVINL float block_rows(Value&& value, int lane, Op&& op) {
    const bool odd = lane & 1, b1 = lane & 2, b2 = lane & 4, b3 = lane & 8;
    float s[8], t[4], u[2];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float even_row = value(2 * i), odd_row = value(2 * i + 1);
        s[i] = op(odd ? odd_row : even_row, swap1(odd ? even_row : odd_row));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = op(b1 ? s[2 * i + 1] : s[2 * i], swap2(b1 ? s[2 * i] : s[2 * i + 1]));
#pragma unroll
    for (int i = 0; i < 2; ++i) u[i] = op(b2 ? t[2 * i + 1] : t[2 * i], __shfl_xor(b2 ? t[2 * i] : t[2 * i + 1], 4, 64));
    const float v = op(b3 ? u[1] : u[0], __shfl_xor(b3 ? u[0] : u[1], 8, 64));
    return op(v, __shfl_xor(v, 16, 64));
}

// What stands for a block among the exponents.  scale_of_row, sb: the scales of the rows and of the column; live: the column is
// one of the block's (others' coefficients are zeros, and no reason to look twice).
template <class Scales>
DEVINL int coef_block_exponent(const float (&c)[16], Scales&& scale_of_row, float sb, bool live, int lane) {
    constexpr float kTiny = 0x1p-100f;
    float top = 0.f, least = INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float t = fabsf(c[r] * scale_of_row(r));
        top = fmaxf(top, t);
        least = fminf(least, t);
    }
    const int col = pow2_exponent(sb);
    const uint32_t bits = wave_max_bits(ldexpf(top, col));
    const int e = ((int)(bits >> 23) - 127 - 14 + 3) & ~3;
    const bool fits = bits >= __float_as_uint(kTiny) && bits < __float_as_uint(0x1p100f);
    if (__builtin_expect(fits && !__ballot(live && (least < kTiny || ldexpf(least, col - e) < kSmallCoef)), 1)) return e;
    // seldom (zeros among them: rows behind a block's last head)
    asm volatile("" ::: "memory");  // (scales that stand in LDS are read again, not kept)
    uint64_t gone = 0u;  // a coefficient that is not zero, but is with its scales, or nearly
    float most = 0.f;
    const auto larger = [](float a, float b) { return fmaxf(a, b); };
    const float row = block_rows([&](int r) __attribute__((always_inline)) {
        const float t = fabsf(c[r] * scale_of_row(r)), x = ldexpf(t, col - e);
        gone |= __ballot(c[r] != 0.f && !(t >= kTiny));
        most = fmaxf(most, x);
        return x;
    }, lane, larger);
    if (!fits) return (__ballot(top != 0.f) | gone) ? kDirect : kNoExponent;
    most = fmaxf(most, __shfl_xor(most, 32, 64));
    auto below = [&](float limit) { return __ballot((row != 0.f && row < limit) || (most != 0.f && most < limit)); };
    if (gone | below(kSmallCoef / (float)(1 << kSmallShift))) return kDirect;
    return e | (below(kSmallCoef) ? 1 : 0);
}

// The block to its place in the matrix of halves, block corner (m0, n0) of block d; `word`: coef_block_exponent's.
// Neighbouring lanes swap values so that a lane stores two columns of one row as one word.  For L2 also the block's row
// sums and column sums (zeros where the direct form takes the block).
template <int DIST, class Scales>
DEVINL void store_coef_block(float (&c)[16], Scales&& scale_of_row, float sb, int word, const SplitCoef& p, int d, int m0, int n0,
                             int lane) {
    const int Bp = p.Bp, Tp = p.Tp;
    if (m0 >= Bp || n0 >= Tp) return;
    const int cl = lane & 31, hl = lane >> 5;
    const bool odd = lane & 1, empty = word >= kNoExponent;
    if (lane == 0) p.exponent[((size_t)d * (Bp >> 5) + (m0 >> 5)) * (Tp >> 5) + (n0 >> 5)] = word;
    if (DIST == DIST_L2) {
        const float v = block_rows([&](int r) { return c[r]; }, lane, [](float a, float b) { return a + b; });
        const int r = lane & 15;
        if (!(lane & 16))
            p.rowpart[((size_t)d * Bp + m0 + 8 * (r >> 2) + 4 * hl + (r & 3)) * (Tp >> 5) + (n0 >> 5)] = empty ? 0.f : v;
        float col = 0.f;
#pragma unroll
        for (int k = 0; k < 16; ++k) col += c[k];
        col += __shfl_xor(col, 32, 64);
        if (lane < 32) p.colpart[((size_t)d * (Bp >> 5) + (m0 >> 5)) * Tp + n0 + lane] = empty ? 0.f : col;
        __builtin_amdgcn_sched_barrier(0);  // (from here on no sums beside the coefficients)
    }
    if (empty) return;  // (the backward leaves the block's halves alone)
    asm volatile("" ::: "memory");
    const int shift = pow2_exponent(sb) - (word & ~3), pitch = half_pitch(Tp);
    const size_t corner = ((size_t)d * Bp + m0) * pitch + (size_t)(n0 >> 5) * kHalfBytes;
    const uint32_t off = (uint32_t)((4 * hl + odd) * pitch + (cl & ~1) * 2);
    auto pack = [&](char* base, auto one_by_one, auto&& value) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (decltype(one_by_one)::value) __builtin_amdgcn_sched_barrier(0);
            // row 2 i + odd of this lane's half
            const float even_row = value(2 * i), odd_row = value(2 * i + 1);
            const float got = swap1(odd ? even_row : odd_row);
            const float x = odd ? got : even_row, y = odd ? odd_row : got;
            uint32_t w[2];
            split2_f16(x, y, w);
            char* const q = base + (size_t)(8 * (i >> 1) + 2 * (i & 1)) * pitch;
#pragma unroll
            for (int k = 0; k < 2; ++k) *reinterpret_cast<uint32_t*>(q + off + 64 * k) = w[k];
        }
    };
    auto scaled = [&](int r) __attribute__((always_inline)) { return ldexpf(c[r] * scale_of_row(r), shift); };
    pack(p.coefp + corner, std::false_type{}, scaled);
    if (__builtin_expect(!(word & 1), 1)) return;
    // seldom: once more, in two parts (and from the coefficients, instead of what would have to be kept for it)
    auto apart = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(c[r])::"memory");
    };
    apart();
    pack(p.coefp + corner, std::true_type{}, [&](int r) { const float v = scaled(r); return fabsf(v) < kSmallCoef ? 0.f : v; });
    apart();
    pack(p.small + corner, std::true_type{}, [&](int r) { const float v = scaled(r); return fabsf(v) < kSmallCoef ? ldexpf(v, kSmallShift) : 0.f; });
}

// The same from float32 coefficients in memory (the losses that are formed row by row): one wave
// per 32 x 32 block.
template <int DIST>
__global__ __launch_bounds__(256) void k_coef_halves(ScoreShape sh, const float* __restrict__ coef, const float* __restrict__ scale,
                                                     int n_head, SplitCoef p) {
    const int lane = threadIdx.x & 63, MT = p.Bp >> 5, NT = p.Tp >> 5;
    const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int d = g / (MT * NT), mt = (g - d * MT * NT) / NT, nt = g % NT;
    if (d >= sh.S || 32 * nt >= tail_limit(sh.tcount, d, sh.T, sh.tpad)) return;
    const int n_live = sh.tcount ? (int)sh.tcount[d] : sh.T;
    const float* src = coef + (size_t)d * sh.B * sh.T;
    const bool near = p.exponent[((size_t)d * MT + mt) * NT + nt] == kDirect;  // as the forward left it
    const int n = 32 * nt + (lane & 31);
    const float sb = scale[n_head + d * sh.T + min(n, sh.T - 1)];
    float c[16], sa[16];
    auto row = [&](int r) __attribute__((always_inline)) { return 32 * mt + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); };
#pragma unroll
    for (int r = 0; r < 16; ++r) {  // all loads in one go: past the last row and column those of the last
        const int m = min(row(r), sh.B - 1);
        sa[r] = scale[d * sh.B + m];
        c[r] = src[(size_t)m * sh.T + min(n, sh.T - 1)];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if (row(r) >= sh.B) sa[r] = 0.f;
        if (row(r) >= sh.B || n >= sh.T) c[r] = 0.f;
    }
    auto scale_a = [&](int r) __attribute__((always_inline)) { return sa[r]; };
    store_coef_block<DIST>(c, scale_a, sb, near ? kDirect : coef_block_exponent(c, scale_a, sb, n < n_live, lane), p, d, 32 * mt, 32 * nt, lane);
}

// --------------------------------------------------------------------------
// forward

// (kCancelRatio, kNearRatio: kge_loss.h)
template <int DIST, int OM, class Tile>
__global__ __launch_bounds__(Tile::threads) __attribute__((amdgpu_waves_per_eu(Tile::EU, Tile::EU))) void k_split_fwd(SplitFwd p) {
    constexpr int TM = Tile::TM, TN = Tile::TN, WM = Tile::WM, WN = Tile::WN;
    using P = SplitProduct<RowTile<TM, 2>, RowTile<TN, 2>, Tile>;
    __shared__ __attribute__((aligned(16))) char smem[P::kLds];
    __shared__ float na_s[TM], nb_s[TN], sa_s[TM], sb_s[TN], mult_s[TN], red[WM * WN];
    __shared__ __attribute__((aligned(16))) uint32_t label_s[TM];
    __shared__ int n_redo;
    const ScoreShape& sh = p.sh;
    const int B = sh.B, T = sh.T, Kp = p.rows.Kp;
    const TileId tile = xcd_tile((T + TN - 1) / TN, (B + TM - 1) / TM, sh.S);
    const int d = tile.z, m0 = tile.y * TM, n0 = tile.x * TN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tid = threadIdx.x, lane = tid & 63;
    const int t_live = tail_limit(sh.tcount, d, T, sh.tpad);
    if (n0 >= t_live) {  // merged tails: the block has no such column
        if (OM == 0 && tid == 0) p.loss_part[(size_t)d * (tile.gx * tile.gy) + tile.y * tile.gx + tile.x] = 0.f;
        return;
    }
    const int n_live = sh.tcount ? (int)sh.tcount[d] : T;
    const int a_row = d * B, b_row = p.rows.n_head + d * T;
    const int pitch = half_pitch(Kp);
    const char* a = p.rows.halves + (int64_t)(a_row + m0) * pitch;
    const char* b = p.rows.halves + (int64_t)(b_row + n0) * pitch;
    floatx16 big, small;
    P::run(smem, a, pitch, kHalfBytes, b, pitch, kHalfBytes, Kp / 32, 0, big, small, lane, wave, [&]() __attribute__((always_inline)) {
        for (int i = tid; i < TM; i += Tile::threads) {
            if (DIST == DIST_L2) na_s[i] = p.rows.norm[a_row + m0 + i];
            sa_s[i] = m0 + i < B ? p.rows.scale[a_row + m0 + i] : 0.f;  // (no row that counts has scale 0)
            if (OM == 0) label_s[i] = m0 + i < B ? p.clabel[d * B + m0 + i] : 0u;
        }
        for (int i = tid; i < TN; i += Tile::threads) {
            if (DIST == DIST_L2) nb_s[i] = p.rows.norm[b_row + n0 + i];
            sb_s[i] = n0 + i < T ? p.rows.scale[b_row + n0 + i] : 0.f;
            if (OM == 0) mult_s[i] = n0 + i < T ? (sh.tmult ? sh.tmult[(size_t)d * T + n0 + i] : 1.f) : 0.f;
        }
    }, [](int) { return true; });

    // epilogue.  Register r of lane l holds row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
    const int mb = 32 * (wave / WN), nbk = 32 * (wave % WN);  // the wave's block's corner in the tile
    const int lane1 = (int)lane_here(), tid1 = 64 * wave + lane1, cl = lane1 & 31, hl = lane1 >> 5;
    const float Tn = (float)T;
    const float w_pos = uniform_f32(0.5f * Tn), w_neg = uniform_f32((0.5f * Tn) / (float)(T - 1));
    const float inv_norm = uniform_f32(1.f / ((float)sh.S * (float)B * Tn));
    // score = base + sign * (distance or product); a coefficient is sign * dL/dscore
    const bool plain = score_is_distance_value(sh.score_fn);
    const float score_sign = plain ? 1.f : -1.f, score_base = plain ? 0.f : sh.gamma;
    const float coef_scale = uniform_f32(inv_norm * sh.loss_scale * score_sign);
    const int Bp = p.out.Bp, Tp = p.out.Tp, MT = Bp >> 5, NT = Tp >> 5;
    float loss_acc = 0.f;
    const int n = n0 + nbk + cl;
    // columns behind a block's distinct tails repeat its first row, the most popular one more
    // often than not: no pair of theirs is worth a second look
    const bool col_counts = n < n_live;
    const float sb = sb_s[nbk + cl];
    float val[16];
    const float* const sa = sa_s + mb + 4 * hl;
    auto scale_a = [&](int r) __attribute__((always_inline)) { return sa[8 * (r >> 2) + (r & 3)]; };
    const float nb = DIST == DIST_L2 ? nb_s[nbk + cl] : 0.f;
    const float* const na = na_s + mb + 4 * hl;
    auto norms = [&](int r) __attribute__((always_inline)) { return na[8 * (r >> 2) + (r & 3)] + nb; };
    uint64_t redo = 0u;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float product = fmaf(small[r], kHalfStep, big[r]);
        if (DIST == DIST_L2) {
            const float ns = norms(r);
            val[r] = fmaf(product, -2.f * sb * scale_a(r), ns);
            redo |= __ballot(!(val[r] > kCancelRatio * ns));
        } else {
            val[r] = product * scale_a(r) * sb;
            redo |= __ballot(!(fabsf(val[r]) < INFINITY));
        }
    }
    bool flagged = false;
    // rare: pairs are recomputed directly, half a wave to a pair, by all of the workgroup (a popular row's
    // come together in one wave's block): those that cancelled, and those that are not finite (an infinity's
    // second half is NaN; a wide row's scale is).  Pairs that do not count, a NaN among them, get any finite value.
    if (__builtin_expect(__syncthreads_or(redo != 0u), 0)) {
        float* const result = reinterpret_cast<float*>(smem);  // [TM][TN]; the tiles are no longer needed
        uint16_t* const list = reinterpret_cast<uint16_t*>(smem + TM * TN * 4);
        static_assert(TM * TN * 6 <= P::kLds, "the tile's pairs as a list and as results");
        if (tid1 == 0) n_redo = 0;
        __syncthreads();
        uint32_t cancel = 0u, near = 0u;
        const int at = (mb + 4 * hl) * TN + nbk + cl;  // of register 0
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const bool live = col_counts && scale_a(r) != 0.f;
            if (!live) val[r] = 0.f;
            else if (DIST == DIST_L2 ? !(val[r] > kCancelRatio * norms(r)) : !(fabsf(val[r]) < INFINITY)) cancel |= 1u << r;
            result[at + (8 * (r >> 2) + (r & 3)) * TN] = val[r];  // (their registers are wanted meanwhile)
        }
        for (uint32_t left = cancel; left; left &= left - 1) {
            const int r = __ffs((int)left) - 1;
            list[atomicAdd(&n_redo, 1)] = (uint16_t)(at + (8 * (r >> 2) + (r & 3)) * TN);
        }
        __syncthreads();
#pragma unroll 1
        for (int q = tid1 >> 5; q < n_redo; q += Tile::threads / 32) {
            const int pos = list[q];
            float part = 0.f;
#pragma unroll 1
            for (int k = (lane1 & 31) * 8; k < Kp; k += 256) {
                Row8 x, y;
                x.load(p.rows, a_row + m0 + pos / TN, k);
                y.load(p.rows, b_row + n0 + pos % TN, k);
                auto add = [&](auto wide) __attribute__((always_inline)) {
                    static_for<8>([&](auto I) {
                        const float u = x.template value<I, decltype(wide)::value>(), v = y.template value<I, decltype(wide)::value>();
                        part = DIST == DIST_L2 ? fmaf(u - v, u - v, part) : fmaf(u, v, part);
                    });
                };
                // (L2 recomputes pairs every day, and without the look 16 blocks of 256 x 1536 take 34.3 us instead of 33.4; dot does not, and the
                // second copy's code costs it 0.7 of 7.0, 4 blocks of 200 x 268, D = 100)
                if (DIST == DIST_L2 && __builtin_expect(!__ballot(is_wide(x.scale) || is_wide(y.scale)), 1)) add(std::false_type{});
                else add(std::true_type{});
            }
            part += swap1(part);
            part += swap2(part);
            part += mirror8(part);
            part += mirror16(part);
            part += __shfl_xor(part, 16, 64);
            if ((lane1 & 31) == 0) result[pos] = part;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            val[r] = result[at + (8 * (r >> 2) + (r & 3)) * TN];
            if (DIST == DIST_L2 && ((cancel >> r) & 1u) && val[r] < kNearRatio * norms(r)) near |= 1u << r;
        }
        for (uint32_t left = cancel; left; left &= left - 1) {  // (a wide row's pairs)
            const int r = __ffs((int)left) - 1;
            if (is_wide(sa[8 * (r >> 2) + (r & 3)]) || is_wide(sb)) near |= 1u << r;
        }
        flagged = __ballot(near != 0u) != 0;
        if (OM == 0)
#pragma unroll
            for (int r = 0; r < 16; ++r) loss_acc += val[r] - val[r];  // a pair that is not finite shows in the loss
    }
    if (OM != 0) {  // raw scores (and distances), and which blocks the direct form is to take
        if (lane1 == 0 && m0 + mb < Bp && n0 + nbk < Tp)
            p.out.exponent[((size_t)d * MT + ((m0 + mb) >> 5)) * NT + ((n0 + nbk) >> 5)] = flagged ? kDirect : kNoExponent;
        float* const out = p.coef + (size_t)d * B * T;
        float* const out_d = (DIST == DIST_L2 && p.dist) ? p.dist + (size_t)d * B * T : nullptr;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + mb + 8 * (r >> 2) + 4 * hl + (r & 3);
            const float dist = DIST == DIST_L2 ? __builtin_amdgcn_sqrtf(val[r]) : val[r];  // (never negative; a NaN stays one)
            if (m < B && n < T) {
                out[(size_t)m * T + n] = score_is_distance_value(sh.score_fn) ? dist : sh.gamma - dist;
                if (out_d) out_d[(size_t)m * T + n] = dist;
            }
        }
        return;
    }
    // a column's negatives: mult of them, or one less where one is the row's label (src/poplar_kge.cpp:615-636)
    const float mult = mult_s[nbk + cl], w_all = mult * w_neg, w_less = (mult - 1.f) * w_neg;
    const bool whole = m0 + mb + 32 <= B && n0 + nbk + 32 <= T;
    float c[16];
    asm volatile("" ::: "memory");  // what stands in LDS is read again, not kept in registers
#pragma unroll
    for (int g = 0; g < 16; g += 4) {  // four rows at a time: their chains of dependent instructions side by side
        const uint4 label4 = *reinterpret_cast<const uint4*>(&label_s[mb + 4 * hl + 2 * g]);
        const uint32_t label[4] = {label4.x, label4.y, label4.z, label4.w};
        float dist[4], term[4], ds[4];
        LogSigmoid z[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            dist[r] = DIST == DIST_L2 ? __builtin_amdgcn_sqrtf(val[g + r]) : val[g + r];  // (never negative; a NaN stays one)
            z[r] = LogSigmoid(fmaf(dist[r], score_sign, score_base));
            const float w = (uint32_t)n == label[r] ? w_less : w_all;
            term[r] = -(w * z[r].minus_value());
            ds[r] = w * z[r].minus_grad();
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool pos = (uint32_t)n == label[r];
            if (__ballot(pos)) {  // one pair of a positive's row
                term[r] -= pos ? w_pos * z[r].plus_value() : 0.f;
                ds[r] -= pos ? w_pos * z[r].plus_grad() : 0.f;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = ds[r] * coef_scale;
            if (DIST == DIST_L2) v = dist[r] != 0.f ? v * __builtin_amdgcn_rcpf(dist[r]) : 0.f;
            if (!whole && !(scale_a(g + r) != 0.f && sb != 0.f)) term[r] = v = 0.f;
            loss_acc += term[r];
            c[g + r] = v;
        }
        __builtin_amdgcn_sched_barrier(0);  // no more rows' intermediate values at once
    }
    asm volatile("" ::: "memory");
    const int word = flagged ? kDirect : coef_block_exponent(c, scale_a, sb, col_counts, lane1);
    if (word == kDirect) {  // the backward takes this block in the direct form, from the coefficients as they are
        char* const out = (char*)(p.coef + ((size_t)d * B + m0 + mb) * T + n0 + nbk);
        const uint32_t off = (uint32_t)(4 * hl * T + cl) * 4;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if (scale_a(r) != 0.f && sb != 0.f) *reinterpret_cast<float*>(out + (size_t)(8 * (r >> 2) + (r & 3)) * T * 4 + off) = c[r];
        }
    }
    store_coef_block<DIST>(c, scale_a, sb, word, p.out, d, m0 + mb, n0 + nbk, lane1);
    if (OM == 0) {
        loss_acc = wave_sum(loss_acc);
        if (lane1 == 0) red[wave] = loss_acc;
        __syncthreads();
        if (tid1 == 0) {
            float tot = 0.f;
#pragma unroll
            for (int w = 0; w < WM * WN; ++w) tot += red[w];
            p.loss_part[(size_t)d * (tile.gx * tile.gy) + tile.y * tile.gx + tile.x] = tot * inv_norm;
        }
    }
}

// --------------------------------------------------------------------------
// backward.  out[i, k] = sum_j c[i, j] phi(self[i, k], other[j, k]), phi = other (dot) or self - other
// (L2: self[i, k] sum_j c[i, j] - the product).  Head side: i = heads, the coefficient rows lie along
// the contraction.  Tail side: i = tails, they lie across it.  `other` always lies across it.
//
// The sub-blocks' own scales: a wave's sums stand in that of the last slab, and are brought to the next one's where that
// differs.  Sums a long way above a slab's scale would not fit it, so a pass takes the slabs within 2^32 of the wave's
// first.  What that leaves, the matrix of small coefficients and the sub-blocks of the direct form are added to the
// results by passes of their own.  They are rare (a table of ordinary rows has none), and all of their code stands behind the main
// pass's, from the kernel's arguments on: in one loop with it, it cost that registers and, through what lay between its
// instructions, 1.5 of 8 us (4 blocks of 200 x 268, D = 100).
constexpr int kMainPass = 8, kSmallPass = 24;  // pass: that of the slabs around the wave's first, plus the distance / 2^64
constexpr uint32_t kDirectPass = 1u << 31;

template <int DIST, bool SIDE_B, class Tile>
struct SplitBwdTile {
    static constexpr int TM = Tile::TM, TN = Tile::TN, WM = Tile::WM, WN = Tile::WN, kSums = Tile::threads / TM;
    using TA = std::conditional_t<SIDE_B, ColTile<TM, 2>, RowTile<TM, 2>>;
    using P = SplitProduct<TA, ColTile<TN, 2>, Tile>;
    const SplitBwd& p;
    char* const smem;
    float* const csum_s;
    int* const exp_s;
    const int tid, d, i0, kt0;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = (wave / WN) * (TM / WM), wn = (wave % WN) * (TN / WN);
    const int B = p.B, T = p.T, Dp = p.rows.Dp, Kp = p.rows.Kp, Bp = p.in.Bp, Tp = p.in.Tp, MT = Bp >> 5, NT = Tp >> 5;
    const int pitch = half_pitch(Kp), coef_pitch = half_pitch(Tp);
    const int t_live = tail_limit(p.tcount, d, T, p.tpad);  // merged tails: the block's live columns
    const int n_self = SIDE_B ? t_live : B, n_other = SIDE_B ? B : t_live, n_slab = (n_other + 31) >> 5;
    const int self0 = SIDE_B ? p.rows.n_head + d * T : d * B, other0 = SIDE_B ? d * B : p.rows.n_head + d * T;

    DEVINL SplitBwdTile(const SplitBwd& p_, char* smem_, float* csum, int* exps, int tid_, int d_, int tile_x, int tile_y)
        : p(p_), smem(smem_), csum_s(csum), exp_s(exps), tid(tid_), d(d_), i0(tile_y * TM), kt0(tile_x * TN) {}

    // a sub-block's exponent: of the self rows' group st and of slab ot
    DEVINL int exponent_of(int st, int ot) const { return p.in.exponent[(size_t)d * MT * NT + (SIDE_B ? (size_t)ot * NT + st : (size_t)st * NT + ot)]; }

    // MAIN: the main pass, what this wave leaves to `todo`; or pass `pass`, added to the results
    template <bool MAIN>
    DEVINL void sums(int pass, uint32_t& todo) const {
        const size_t corner = (size_t)d * Bp * coef_pitch + (SIDE_B ? (size_t)(i0 >> 5) * kHalfBytes : (size_t)i0 * coef_pitch);
        const char* const a = (MAIN || pass < 16 ? p.in.coefp : p.in.small) + corner;
        const char* const b = p.rows.halves + (int64_t)other0 * pitch + (size_t)(kt0 >> 5) * kHalfBytes;
        const bool alive = i0 + wm < n_self;  // any of the wave's rows
        const int st0 = min((i0 + wm) >> 5, (SIDE_B ? NT : MT) - 1);  // (rows past the last are dropped)
        int exp_reg;  // of slab 64 n + lane
        auto load_exps = [&](int slab0) __attribute__((always_inline)) { exp_reg = exponent_of(st0, min(slab0 + lane, n_slab - 1)); };
        constexpr int kNone = kDirect + 4;
        int first = kNone, now = kNone;  // the wave's first slab's exponent; what the sums are in
        floatx16 big, small;
        P::run(smem, a, coef_pitch, SIDE_B ? (size_t)32 * coef_pitch : kHalfBytes, b, pitch, (size_t)32 * pitch, n_slab, n_other, big, small, lane, wave,
               [&]() __attribute__((always_inline)) {
                   load_exps(0);
                   if (!MAIN) return;
                   if (tid < TM) exp_s[tid] = pow2_exponent(p.rows.scale[self0 + i0 + tid]);
                   if (DIST != DIST_L2) return;
                   // the self rows' coefficient sums, from the sub-blocks' in a fixed order: kSums threads to a row, four
                   // loads of each under way
                   const int i = tid % TM, n = SIDE_B ? MT : n_slab;
                   if (i0 + i < (SIDE_B ? Tp : Bp)) {
                       const float* part = SIDE_B ? p.in.colpart + (size_t)d * MT * Tp + i0 + i : p.in.rowpart + ((size_t)d * Bp + i0 + i) * NT;
                       const size_t step = SIDE_B ? Tp : 1;
                       float s = 0.f;
                       for (int q = tid / TM; q < n; q += 4 * kSums) {
                           float v[4];
#pragma unroll
                           for (int x = 0; x < 4; ++x) v[x] = q + x * kSums < n ? part[(q + x * kSums) * step] : 0.f;
                           s += (v[0] + v[1]) + (v[2] + v[3]);
                       }
                       csum_s[tid] = s;
                   } else {
                       csum_s[tid] = 0.f;
                   }
               },
               [&](int slab) __attribute__((always_inline)) {
                   if (slab && !(slab & 63)) load_exps(slab);
                   const int word = __builtin_amdgcn_readlane(exp_reg, slab & 63);
                   if (MAIN && word == now) return true;  // the rule
                   if (!alive || word >= kNoExponent) {
                       if (MAIN && alive && word == kDirect) todo |= kDirectPass;
                       return false;
                   }
                   int e = word & ~3;
                   if (first == kNone) first = e;
                   const int here = kMainPass + ((e - first + 32) >> 6), of_small = kSmallPass + ((e - kSmallShift - first + 32) >> 6);
                   if (MAIN) {
                       if (word & 1) todo |= 1u << of_small;
                       if (here != kMainPass) {
                           todo |= 1u << here;
                           return false;
                       }
                   } else {
                       if (pass < 16 ? pass != here : !(word & 1) || pass != of_small) return false;
                       if (pass >= 16) e -= kSmallShift;
                   }
                   if (now != kNone) {
                       const float by = __uint_as_float((uint32_t)(127 + now - e) << 23);
#pragma unroll
                       for (int r = 0; r < 16; ++r) {
                           big[r] *= by;
                           small[r] *= by;
                       }
                   }
                   now = e;
                   return true;
               });
        const int lane1 = (int)lane_here(), cl = lane1 & 31, hl = lane1 >> 5;
        // the self rows' own scales leave the sums
#pragma unroll
        for (int r = 0; r < 16; ++r)
            big[r] = ldexpf(fmaf(small[r], kHalfStep, big[r]),
                                  (now == kNone ? 0 : now) - exp_s[wm + 8 * (r >> 2) + 4 * hl + (r & 3)]);
        const char* const self = p.rows.halves + (int64_t)(self0 + i0) * pitch;
        // neighbouring lanes swap values: a lane stores two columns of one row
        const bool odd = lane1 & 1;
        float* const out = p.grad + (size_t)(self0 + i0) * Dp;
        const int k = kt0 + wn + (cl & ~1);
        if (k >= Dp) return;
        // (a row: the wave's part, in scalars, and the lane's, in one offset for all of them)
        const uint32_t in_off = (uint32_t)((4 * hl + odd) * pitch + (k >> 5) * kHalfBytes + (k & 31) * 2);
        const uint32_t lost_off = (uint32_t)((4 * hl + odd) * (Kp >> 5) + (k >> 5)) * 4;
        const uint32_t out_off = (uint32_t)((4 * hl + odd) * Dp + k) * 4;
        auto wave_row = [&](int i) __attribute__((always_inline)) { return wm + 8 * (i >> 1) + 2 * (i & 1); };
        constexpr bool kSelf = MAIN && DIST == DIST_L2;
        uint32_t w[kSelf ? 8 : 1][3];
        if (kSelf)
#pragma unroll
            for (int i = 0; i < 8; ++i) {  // all loads before any use, rows past the last among them
                const char* const row = self + (int64_t)wave_row(i) * pitch;
#pragma unroll
                for (int q = 0; q < 2; ++q) w[i][q] = *reinterpret_cast<const uint32_t*>(row + in_off + 64 * q);
                w[i][2] = *reinterpret_cast<const uint32_t*>((const char*)(p.rows.lost + (int64_t)(self0 + i0 + wave_row(i)) * (Kp >> 5)) + lost_off);
            }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float got = swap1(odd ? big[2 * i] : big[2 * i + 1]);
            float x = odd ? got : big[2 * i], y = odd ? big[2 * i + 1] : got;
            const int row = wave_row(i) + 4 * hl + odd;
            if (kSelf) {
                const f16x2 h = __builtin_bit_cast(f16x2, w[i][0]), l = __builtin_bit_cast(f16x2, w[i][1]);
                float sum = csum_s[row];
#pragma unroll
                for (int q = 1; q < kSums; ++q) sum += csum_s[row + q * TM];
                sum = ldexpf(sum, exp_s[row]);
                // (every bit of the self row: against this product the other one is small)
                const uint32_t lost = w[i][2] >> lost_at(k);
                x = join_lost(h.x, l.x, lost & 1u) * sum - x;
                y = join_lost(h.y, l.y, (lost >> 8) & 1u) * sum - y;
                if (exp_s[row] == kWideExponent) x = y = 0.f;  // (all of it by the direct form)
            }
            if (i0 + row >= n_self) continue;
            float2* const at = reinterpret_cast<float2*>((char*)(out + (size_t)wave_row(i) * Dp) + out_off);
            *at = MAIN ? make_float2(x, y) : DIST == DIST_L2 ? make_float2(at->x - x, at->y - y) : make_float2(at->x + x, at->y + y);
        }
    }

    // the direct form: c (self - other), or c other, one pair after the other as the reference codelet does (sub-blocks in
    // which some pair is nearly identical, or coefficients that halves do not hold), added to what the workgroup has
    // stored.  A wave takes four rows at a time, a lane a column.
    DEVINL void direct() const {
        static_assert(TN == 64, "a lane per column");
        constexpr int kRows = 4;  // of a slab under way (a divisor of 32)
        const float* const cf = p.coef + (size_t)d * B * T;
        const int lane1 = (int)lane_here(), k = min(kt0 + lane1, Dp - 1);
        auto lane_value = [&](float v, int l) __attribute__((always_inline)) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
        for (int i = i0 + 4 * wave; i < min(i0 + TM, n_self); i += 4 * WM * WN) {
            float add[4] = {0.f, 0.f, 0.f, 0.f};
            int row[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) row[x] = min(i + x, n_self - 1);
            bool any = false;
            for (int ot = 0; ot < n_slab; ++ot) {
                if (exponent_of(i >> 5, ot) != kDirect) continue;
                any = true;
                // the slab's scales, and behind them those of the self rows
                const float scales = p.rows.scale[lane1 < 32 ? other0 + min(32 * ot + lane1, n_other - 1) : self0 + min(i + (lane1 & 3), n_self - 1)];
                float sv[4];
                Row1 raw_self[4];
#pragma unroll
                for (int x = 0; x < 4; ++x) raw_self[x].load(p.rows, self0 + row[x], k, lane_value(scales, 32 + x));
#pragma unroll
                for (int x = 0; x < 4; ++x) sv[x] = raw_self[x].value(k, lane_value(scales, 32 + x));
                const int n = min(32, n_other - 32 * ot);
                float c[4];  // of the slab's row `lane`, zero past the last
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const int j = 32 * ot + min(lane1, n - 1);
                    c[x] = SIDE_B ? cf[(size_t)j * T + row[x]] : cf[(size_t)row[x] * T + j];
                }
#pragma unroll
                for (int x = 0; x < 4; ++x) c[x] = lane1 < n ? c[x] : 0.f;
#pragma unroll 1
                for (int j0 = 0; j0 < n; j0 += kRows) {
                    Row1 raw[kRows];
                    int j[kRows];
#pragma unroll
                    for (int y = 0; y < kRows; ++y) {
                        j[y] = min(j0 + y, n - 1);
                        raw[y].load(p.rows, other0 + 32 * ot + j[y], k, lane_value(scales, j[y]));
                    }
#pragma unroll
                    for (int y = 0; y < kRows; ++y) {
                        const float other = raw[y].value(k, lane_value(scales, j[y]));
#pragma unroll
                        for (int x = 0; x < 4; ++x) add[x] = fmaf(lane_value(c[x], j0 + y), DIST == DIST_L2 ? sv[x] - other : other, add[x]);
                    }
                }
            }
            if (!any || kt0 + lane1 >= Dp) continue;
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (i + x < n_self) p.grad[(size_t)(self0 + i + x) * Dp + k] += add[x];
        }
    }
};

// Both sides in one launch: the side whose tiles loop over more rows comes first, for every block, so
// that the long tiles do not start last.  A block's tiles of one side stay together on one XCD.
template <int DIST, class Tile>
__global__ __launch_bounds__(Tile::threads) __attribute__((amdgpu_waves_per_eu(Tile::EU, Tile::EU))) void k_split_bwd(SplitBwd p) {
    constexpr int TM = Tile::TM, TN = Tile::TN;
    using PA = SplitProduct<RowTile<TM, 2>, ColTile<TN, 2>, Tile>;
    __shared__ __attribute__((aligned(16))) char smem[PA::kLds];
    __shared__ float csum_s[Tile::threads];
    __shared__ int exp_s[TM];
    __shared__ uint32_t todo_s;
    // tile L's work: with(its side, its place)
    auto place = [](const SplitBwd& q, int L, auto&& with) __attribute__((always_inline)) {
        const int gx = (q.rows.Dp + TN - 1) / TN, ga = (q.B + TM - 1) / TM, gb = (q.T + TM - 1) / TM;
        const bool heads_first = q.T >= q.B;
        const int n_first = gx * (heads_first ? ga : gb) * q.S;
        if ((L < n_first) == heads_first) with(std::false_type{}, xcd_tile(gx, ga, q.S, heads_first ? L : L - n_first));
        else with(std::true_type{}, xcd_tile(gx, gb, q.S, heads_first ? L - n_first : L));
    };
    uint32_t todo = 0u;
    if (threadIdx.x == 0) todo_s = 0u;  // (the loop's barriers stand between this and what follows it)
    bool ran = false;
    place(p, blockIdx.x, [&](auto side_b, const TileId& t) __attribute__((always_inline)) {
        const SplitBwdTile<DIST, decltype(side_b)::value, Tile> tile(p, smem, csum_s, exp_s, threadIdx.x, t.z, t.x, t.y);
        ran = tile.i0 < tile.n_self;
        if (ran) tile.template sums<true>(kMainPass, todo);
    });
    if (!ran) return;
    if (todo && (threadIdx.x & 63) == 0) atomicOr(&todo_s, todo);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (not __syncthreads: the results' stores are no reason to wait)
    todo = (uint32_t)__builtin_amdgcn_readfirstlane((int)todo_s);
    if (__builtin_expect(!todo, 1)) return;
    // seldom.  Nothing that the main pass has computed is kept for this, nor from one pass for the next.
    auto anew = [&](auto&& with) __attribute__((always_inline)) {
        auto args = (const __attribute__((address_space(4))) uint32_t*)__builtin_amdgcn_kernarg_segment_ptr();
        int L = blockIdx.x, tid = threadIdx.x;
        asm volatile("" : "+s"(args), "+s"(L), "+v"(tid));
        struct Words { uint32_t w[sizeof(SplitBwd) / 4]; } words;
        static_assert(sizeof(Words) == sizeof(SplitBwd));
#pragma unroll
        for (size_t i = 0; i < sizeof(SplitBwd) / 4; ++i) words.w[i] = args[i];
        const SplitBwd q = __builtin_bit_cast(SplitBwd, words);
        place(q, L, [&](auto side_b, const TileId& t) __attribute__((always_inline)) {
            with(SplitBwdTile<DIST, decltype(side_b)::value, Tile>(q, smem, csum_s, exp_s, tid, t.z, t.x, t.y));
        });
    };
    __syncthreads();
#pragma unroll 1
    for (; todo & ~kDirectPass; todo &= todo - 1u) {
        uint32_t none = 0u;
        anew([&](auto&& tile) __attribute__((always_inline)) { tile.template sums<false>(__ffs((int)todo) - 1, none); });
        __syncthreads();  // (of the tiles in LDS, too)
    }
    if (todo) anew([](auto&& tile) __attribute__((always_inline)) { tile.direct(); });
}

// --------------------------------------------------------------------------
// launches

// Which tiles.  128 x 64 read a third less, 64 x 64 are twice as many.  Large tiles are counted as if all tails were distinct (how many
// are, only the device knows).  Launches, us, 64 x 64 and 128 x 64, D = 256, all tails distinct, behind each the large tiles:
// Forward: 32 blocks of 256 x 256 14.6, 15.3 (256); 40 of 256 x 240 17.4, 19.2 (320); 48 18.5, 20.5 (384); 64 of 256 x 256 21.9, 23.6,
// 32 of 256 x 512 21.3, 22.0, 8 of 1024 x 512 20.7, 20.7 (512); 40 of 256 x 480 27.8, 26.1 (640); 16 of 256 x 1536 32.1, 27.8 (768);
// 64 of 256 x 512, 331 distinct, 31.1, 26.9 (1024); 4 of 200 x 268, D = 100, 11.6, 13.1 (40); one of 256 x 64, D = 64, 9.1, 10.1 (2).
// Heads that fill half of their large tiles: 48 of 129 x 672, D = 100, 27.0, 30.6 (1056).
// Backward: 6 of 1024 x 510 27.5, 31.4 (288); 8 of 1024 x 512 25.4, 28.4 (384); 32 of 256 x 256 18.3, 17.4 (512); 32 of 256 x 512
// 32.6, 27.1 (768); 64 of 256 x 256 32.3, 31.1 (1024); 64 of 256 x 512, 331 distinct, 39.8, 40.4 (1536); 4 of 200 x 268 9.8, 11.1 (40).
// Where the contraction is long on one side only, the small ones would be the faster: 16 of 256 x 1536 38.5, 44.0 (896).
static bool large_tiles(const ScoreShape& sh) {
    return (int64_t)sh.S * ((sh.B + 127) / 128) * ((sh.T + 63) / 64) >= 512;
}
static bool large_tiles_bwd(const SplitBwd& p) {
    return (int64_t)p.S * ((p.B + 127) / 128 + (p.T + 127) / 128) * ((p.rows.Dp + 63) / 64) >= 512;
}

int split_fwd_parts(const ScoreShape& sh) {
    const int tm = large_tiles(sh) ? TileLarge::TM : TileSmall::TM;
    return ((sh.T + 63) / 64) * ((sh.B + tm - 1) / tm);
}

template <int DIST, int OM>
static void split_fwd(const SplitFwd& p, hipStream_t stream) {
    const ScoreShape& sh = p.sh;
    if (large_tiles(sh))
        hipLaunchKernelGGL((k_split_fwd<DIST, OM, TileLarge>), tile_grid((sh.T + 63) / 64, (sh.B + 127) / 128, sh.S),
                           dim3(TileLarge::threads), 0, stream, p);
    else
        hipLaunchKernelGGL((k_split_fwd<DIST, OM, TileSmall>), tile_grid((sh.T + 63) / 64, (sh.B + 63) / 64, sh.S),
                           dim3(TileSmall::threads), 0, stream, p);
}
void launch_split_fwd(const SplitFwd& p, bool fused_loss, hipStream_t stream) {
    const bool l2 = p.sh.dist_fn == DIST_L2 && p.sh.score_fn != SCORE_DISTMULT;
    if (l2) fused_loss ? split_fwd<DIST_L2, 0>(p, stream) : split_fwd<DIST_L2, 1>(p, stream);
    else fused_loss ? split_fwd<DIST_DOT, 0>(p, stream) : split_fwd<DIST_DOT, 1>(p, stream);
}

void launch_coef_halves(const ScoreShape& sh, const float* coef, const SplitRows& rows, const SplitCoef& out, hipStream_t stream) {
    const int n = sh.S * (out.Bp / 32) * (out.Tp / 32);
    const bool l2 = sh.dist_fn == DIST_L2 && sh.score_fn != SCORE_DISTMULT;
#define KGE_COEF(D_) \
    hipLaunchKernelGGL(k_coef_halves<D_>, dim3((n + 3) / 4), dim3(256), 0, stream, sh, coef, rows.scale, rows.n_head, out)
    if (l2) KGE_COEF(DIST_L2);
    else KGE_COEF(DIST_DOT);
#undef KGE_COEF
}

template <int DIST, class Tile>
static void split_bwd(const SplitBwd& p, hipStream_t stream) {
    const dim3 grid(((p.rows.Dp + Tile::TN - 1) / Tile::TN) * ((p.B + Tile::TM - 1) / Tile::TM + (p.T + Tile::TM - 1) / Tile::TM) * p.S);
    hipLaunchKernelGGL((k_split_bwd<DIST, Tile>), grid, dim3(Tile::threads), 0, stream, p);
}
void launch_split_bwd(const SplitBwd& p, bool l2, hipStream_t stream) {
    if (large_tiles_bwd(p)) l2 ? split_bwd<DIST_L2, TileLarge>(p, stream) : split_bwd<DIST_DOT, TileLarge>(p, stream);
    else l2 ? split_bwd<DIST_L2, TileSmall>(p, stream) : split_bwd<DIST_DOT, TileSmall>(p, stream);
}

// Where these kernels are taken: L2 and dot of every shape.  (Kernels that split float32 operands into bfloat16 pieces while
// staging took 38 + 55 us for the forward and backward of 64 blocks of 256 x 512, these take 28 + 44; 32 of 256 x 256: 15 + 21
// and 13 + 16.)
bool split_scoring(const ScoreShape& sh) {
    if (sh.use_mfma != 2 || sh.score_fn == SCORE_TRANSH) return false;
    return !(sh.dist_fn == DIST_L1 && sh.score_fn != SCORE_DISTMULT);
}

}  // namespace kge
