// gfx950 kernels of the feature projection (src/poplar_kge.cpp:451-462): hidden = embedding + feature . W
// for the distinct rows, and dW = feature^T . gradient.
//
// Both are float32 products formed from bfloat16 matrix instructions.  A feature stored in 16 bits is
// exactly two bfloat16 pieces (float16: 8 + 3 significant bits) or one (bfloat16), W and the
// gradient are three; the products of pieces below 2^-24 of the result are left out: five, three or
// (float32 features) six instructions per sixteen contraction steps.  The features are read where they
// lie, in the table, and split while they are staged: no dense copy of them is made.
#include "kge_split.h"

#include <algorithm>
#include <cstdint>

namespace kge {

template <int FT> struct Pieces { static constexpr int n = FT == ET_F16 ? 2 : FT == ET_BF16 ? 1 : 3; };

// eight consecutive features, as they lie
template <int FT> struct Raw8 { uint4 v[FT == ET_F32 ? 2 : 1]; };
template <int FT>
DEVINL void load_raw8(Raw8<FT>& r, const char* row, int f, int Fp) {  // features f .. f + 7, zero from Fp on (Fp % 4 == 0, 16-bit: % 8)
    constexpr int half = FT == ET_F32 ? 4 : 8;
#pragma unroll
    for (int h = 0; h < 8 / half; ++h)
        r.v[h] = f + half * h < Fp ? *reinterpret_cast<const uint4*>(row + (size_t)(f + half * h) * (FT == ET_F32 ? 4 : 2))
                                   : make_uint4(0u, 0u, 0u, 0u);
}
// The same without a look at Fp, and zeros from Fp on once they have come.
template <int FT>
DEVINL void load_raw8_whole(Raw8<FT>& r, const char* at) {
#pragma unroll
    for (int h = 0; h < (FT == ET_F32 ? 2 : 1); ++h) r.v[h] = *reinterpret_cast<const uint4*>(at + 16 * h);
}
template <int FT>
DEVINL void clear_raw8_past(Raw8<FT>& r, int f, int Fp) {
    constexpr int half = FT == ET_F32 ? 4 : 8;
#pragma unroll
    for (int h = 0; h < 8 / half; ++h)
        if (f + half * h >= Fp) r.v[h] = make_uint4(0u, 0u, 0u, 0u);
}
// -> piece q of the eight, for every piece
template <int FT>
DEVINL void split_raw8(const Raw8<FT>& r, uint4 (&piece)[Pieces<FT>::n]) {
    if constexpr (FT == ET_BF16) {
        piece[0] = r.v[0];
    } else {
        float x[8];
        if constexpr (FT == ET_F32) {
            const uint32_t w[8] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w, r.v[1].x, r.v[1].y, r.v[1].z, r.v[1].w};
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = __uint_as_float(w[i]);
        } else {
            const uint32_t w[4] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float2 f = __half22float2(*reinterpret_cast<const __half2*>(&w[i]));
                x[2 * i] = f.x; x[2 * i + 1] = f.y;
            }
        }
#pragma unroll
        for (int q = 0; q < Pieces<FT>::n; ++q) {
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                w[i] = pack_bf16(x[2 * i], x[2 * i + 1]);
                if (q + 1 < Pieces<FT>::n) { x[2 * i] -= bf16_lo_f32(w[i]); x[2 * i + 1] -= bf16_hi_f32(w[i]); }
            }
            piece[q] = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

// the products of one sixteen-step: AM accumulators, one fragment column of the other operand,
// smallest terms first.  `low`: where all but the largest term go (acc itself, or accumulators of their own)
template <int PA, int AM>
DEVINL void feature_products(const floatx4 (&fa)[AM][PA], const floatx4 (&fb)[3], floatx16 (&acc)[AM], floatx16 (&low)[AM]) {
    constexpr int n = PA == 3 ? 6 : PA == 2 ? 5 : 3;
    constexpr int qa[6] = {PA == 3 ? 0 : PA == 2 ? 1 : 0, PA == 3 ? 2 : 0, PA == 3 ? 1 : PA == 2 ? 1 : 0, 0, PA == 3 ? 1 : 0, 0};
    constexpr int qb[6] = {PA == 3 ? 2 : PA == 2 ? 1 : 2, PA == 3 ? 0 : PA == 2 ? 2 : 1, PA == 3 ? 1 : 0, 1, 0, 0};
#pragma unroll
    for (int x = 0; x < n; ++x)
#pragma unroll
        for (int m = 0; m < AM; ++m) {
            floatx16& to = x + 1 < n ? low[m] : acc[m];
            to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[m][qa[x]]),
                                                         __builtin_bit_cast(bf16x8, fb[qb[x]]), to, 0, 0, 0);
        }
}

// hidden.  A workgroup of NW waves takes 32 AM rows x 32 NW columns, every wave all of the rows and 32 of
// the columns: with D <= 256 a row's features come from memory once.  W lies as a piece matrix
// (launch_split_matrix) and goes straight into LDS.
template <int FT, int AM, int NW>
struct FeatureFwd {
    static constexpr int PA = Pieces<FT>::n, TM = 32 * AM, TN = 32 * NW, NT = NW * 64;
    using TA = RowTile<TM>;
    using TB = ColTile<TN>;
    static constexpr int kA = PA * TM * 64, kStage = kA + TB::kBytes;
};
template <int FT, int AM, int NW>
DEVINL void feature_fwd_tile(const FeatureArgs& a, const char* __restrict__ wp, int w_pitch, float* __restrict__ hidden,
                             char* const smem, uint32_t* const key_s) {
    using Tile = FeatureFwd<FT, AM, NW>;
    using TA = typename Tile::TA;
    using TB = typename Tile::TB;
    constexpr int PA = Tile::PA, TM = Tile::TM, TN = Tile::TN, NT = Tile::NT;
    constexpr int NC = (TM * 4 + NT - 1) / NT;  // 16-byte chunks of a slab per thread
    // Slabs whose features are asked for together: a row of the table is a round trip of microseconds
    // (and its loads hold up the copies behind them: they return in order), so it is paid once for as
    // many slabs as 96 registers hold, not once per slab (24k rows of 768 float16 features, 256 columns, all
    // in one round: 94 us with a round trip per slab, 60 so).  Wider rows pay it once per such a round: with
    // one chunk per thread 768 16-bit or 384 float32 features, with four a quarter of that.
    constexpr int KS = (FT == ET_F32 ? 12 : 24) / NC;
    constexpr int kA = Tile::kA, kStage = Tile::kStage, kEach = TB::kCopies / NW;
    const int gx = (a.Dp + TN - 1) / TN;
    const int u0 = (int)blockIdx.x / gx * TM, n0 = (int)blockIdx.x % gx * TN;
    const int U = (int)a.counts[0];
    if (u0 >= U) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int i = tid; i < TM; i += NT) key_s[i] = a.uniq_key[min(u0 + i, U - 1)];
    __syncthreads();
    const char* src[NC];
    int dst[NC], kc[NC];
    bool on[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int c = tid + NT * i, row = min(c >> 2, TM - 1);
        on[i] = TM * 4 % NT == 0 || c < TM * 4;
        kc[i] = (c & 3) * 8;
        src[i] = a.feat_base + (int64_t)key_s[row] * a.pitch;
        dst[i] = row * 64 + ((c & 3) ^ ((row >> 2) & 3)) * 16;
    }
    uint32_t off[kEach];
#pragma unroll
    for (int i = 0; i < kEach; ++i) off[i] = TB::source(wave + NW * i, lane, w_pitch);
    const char* const w0 = wp + (size_t)(n0 >> 5) * 192;
    const uint32_t lds0 = lds_address(smem) + kA;
    auto fill = [&](int slab) __attribute__((always_inline)) {
        const char* from = w0 + (size_t)slab * 32 * w_pitch;
#pragma unroll
        for (int i = 0; i < kEach; ++i) lds_copy16(from, off[i], lds0 + (slab & 1) * kStage + (wave + NW * i) * 1024);
    };
    const int n_slab = (a.Fp + 31) / 32;
    fill(0);
    const int k = n0 + 32 * wave + (lane & 31);
    floatx16 acc[AM];
#pragma unroll
    for (int m = 0; m < AM; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = 0.f;
    auto multiply = [&](int slab) __attribute__((always_inline)) {
        const char* ta = smem + (slab & 1) * kStage;
        const char* tb = ta + kA;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            floatx4 fa[AM][PA], fb[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) fb[q] = TB::fragment(tb, q, 32 * wave, ks, lane);
#pragma unroll
            for (int m = 0; m < AM; ++m)
#pragma unroll
                for (int q = 0; q < PA; ++q) fa[m][q] = TA::fragment(ta, q, 32 * m, ks, lane);
            feature_products<PA, AM>(fa, fb, acc, acc);
        }
    };
    // The embeddings: added once, to the finished sums (as what the accumulators start from they would
    // make every instruction of the contraction round at their size, 240 times for 768 float16 features),
    // and all asked for together: up front where they have registers, else under the last slab's products.
    const bool wide = a.emb_etype == ET_F32;
    floatx16 emb[AM];
    auto fetch = [&](auto type) __attribute__((always_inline)) {  // as they lie
        using T = decltype(type);
        const T* const col = reinterpret_cast<const T*>(a.emb_base) + min(k, a.Dp - 1);
#pragma unroll
        for (int m = 0; m < AM; ++m)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint4 key4 = *reinterpret_cast<const uint4*>(&key_s[32 * m + 8 * g + 4 * (lane >> 5)]);
                const uint32_t key[4] = {key4.x, key4.y, key4.z, key4.w};
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const T v = *reinterpret_cast<const T*>(reinterpret_cast<const char*>(col) + (uint64_t)key[r] * (uint32_t)a.pitch);
                    if constexpr (sizeof(T) == 4) emb[m][4 * g + r] = v;
                    else emb[m][4 * g + r] = __uint_as_float(v);
                }
            }
    };
    auto fetch_embeddings = [&]() __attribute__((always_inline)) {
        if (!a.emb_base) {
#pragma unroll
            for (int m = 0; m < AM; ++m)
#pragma unroll
                for (int r = 0; r < 16; ++r) emb[m][r] = 0.f;
        } else if (wide) fetch(float{});
        else fetch(uint16_t{});
    };
    if constexpr (AM <= 2) fetch_embeddings();
    for (int s0 = 0; s0 < n_slab; s0 += KS) {
        // By every thread, with nothing between the loads but a scalar branch, their offsets constants: a register
        // written for the next load's address, or with zeros for lanes that have none, waits until all loads so far
        // are back, and the round trips follow one another (64 and 32 queries' sweeps over 4k rows of 768 features,
        // D = 242, 106, 78: 199, 627 and 373 us a pass with such waits, 186, 592 and 353 without).
        // (The last slab of a row may read up to 28 features behind it: the next row, or the spare rows that the table
        // ends in.)
        Raw8<FT> raw[KS][NC];
        constexpr int kElem = FT == ET_F32 ? 4 : 2;
        const char* from[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i) from[i] = src[i] + (32 * s0 + kc[i]) * kElem;
#pragma unroll
        for (int x = 0; x < KS; ++x) {
            if (s0 + x < n_slab)
#pragma unroll
                for (int i = 0; i < NC; ++i) load_raw8_whole<FT>(raw[x][i], from[i] + 32 * x * kElem);
        }
        static_for<KS>([&](auto xc) __attribute__((always_inline)) {
            constexpr int x = decltype(xc)::value;
            const int slab = s0 + x;
            if (slab >= n_slab) return;
            // (a tile copy was last read two slabs ago, before the barrier of the slab in between)
#pragma unroll
            for (int i = 0; i < NC; ++i)
                if (on[i]) {
                    uint4 piece[PA];
                    clear_raw8_past<FT>(raw[x][i], 32 * slab + kc[i], a.Fp);
                    split_raw8<FT>(raw[x][i], piece);
#pragma unroll
                    for (int q = 0; q < PA; ++q)
                        *reinterpret_cast<uint4*>(smem + (slab & 1) * kStage + q * (TM * 64) + dst[i]) = piece[q];
                }
            wait_copies_and_barrier<0>();
            if (slab + 1 < n_slab) {
                fill(slab + 1);
                multiply(slab);
            }
        });
    }
    if constexpr (AM > 2) fetch_embeddings();
    __builtin_amdgcn_sched_barrier(0);
    multiply(n_slab - 1);
    if (k >= a.Dp) return;
#pragma unroll
    for (int m = 0; m < AM; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int u = u0 + 32 * m + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            const uint16_t raw = (uint16_t)__float_as_uint(emb[m][r]);
            const float e = wide ? emb[m][r] : load1(reinterpret_cast<const char*>(&raw), 0, a.emb_etype);
            if (u < U) hidden[(size_t)u * a.Dp + k] = acc[m][r] + e;
        }
}

// Tile height (in 32 rows) for `rows` rows: the one with the fewest rows per CU over all rounds of workgroups.
__host__ DEVINL uint32_t feature_tiles(uint32_t rows, int t, int gx) { return (rows + 32 * t - 1) / (32 * t) * gx; }
__host__ DEVINL int feature_tile(uint32_t rows, int gx, uint32_t slots) {
    int am = 1;
    uint32_t best = UINT32_MAX;
#pragma unroll
    for (int t = 1; t <= 4; ++t) {
        const uint32_t cost = (feature_tiles(rows, t, gx) + slots - 1) / slots * (2 + 3 * t);  // (a tile's W slabs cost as much as some rows)
        if (cost < best) { best = cost; am = t; }
    }
    return am;
}

// AM = 0: the height is the one for the distinct rows, which only the device knows
template <int FT, int AM, int NW>
__global__ __launch_bounds__(NW * 64) void k_feature_fwd(FeatureArgs a, const char* __restrict__ wp, int w_pitch,
                                                         float* __restrict__ hidden) {
    using Most = FeatureFwd<FT, AM ? AM : 4, NW>;
    __shared__ __attribute__((aligned(16))) char smem[2 * Most::kStage];
    __shared__ __attribute__((aligned(16))) uint32_t key_s[Most::TM];
    if constexpr (AM != 0) {
        feature_fwd_tile<FT, AM, NW>(a, wp, w_pitch, hidden, smem, key_s);
    } else {
        const int am = feature_tile(a.counts[0], (a.Dp + 32 * NW - 1) / (32 * NW), 256 * (8 / NW));
        if (am == 1) feature_fwd_tile<FT, 1, NW>(a, wp, w_pitch, hidden, smem, key_s);
        else if (am == 2) feature_fwd_tile<FT, 2, NW>(a, wp, w_pitch, hidden, smem, key_s);
        else if (am == 3) feature_fwd_tile<FT, 3, NW>(a, wp, w_pitch, hidden, smem, key_s);
        else feature_fwd_tile<FT, 4, NW>(a, wp, w_pitch, hidden, smem, key_s);
    }
}

// dW.  A workgroup takes 32 AM features x 32 NW columns over its share of the rows (the output has
// few tiles: the contraction is split, the parts are added up by the update's kernel).  Both
// operands lie across the contraction and are split while staged.
template <int FT, int AM, int NW>
__global__ __launch_bounds__(NW * 64) void k_feature_grad(FeatureArgs a, const float* __restrict__ grad, int n_split,
                                                          float* __restrict__ part) {
    constexpr int PA = Pieces<FT>::n, TM = 32 * AM, TN = 32 * NW, NT = NW * 64;
    static_assert(TM == 128 || TM == 64, "ColTile");
    constexpr int NA = (32 * TM / 8 + NT - 1) / NT, NB = 32 * TN / 4 / NT;
    using TA = ColTile<TM>;
    using TB = ColTile<TN>;
    constexpr int kA = PA * 32 * TM * 2, kStage = kA + TB::kBytes;
    __shared__ __attribute__((aligned(16))) char smem[2 * kStage];
    const int gx = (a.Dp + TN - 1) / TN, gy = (a.Fp + TM - 1) / TM;
    const int split = (int)blockIdx.x / (gx * gy), t = (int)blockIdx.x % (gx * gy), f0 = t / gx * TM, n0 = t % gx * TN;
    const int U = (int)a.counts[0];
    const int share = ((U + n_split - 1) / n_split + 31) & ~31;
    const int ub = split * share, ue = min(U, ub + share), n_slab = ue > ub ? (ue - ub + 31) / 32 : 0;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the small terms in accumulators of their own: the large ones round once per sixteen rows, not five times
    // (dW of 256 rows of 768 float16 features, against float64: 1.95e-7 off with one set, 1.5e-7 with two,
    // most of it the gradient's; the time is the same, 60 us for 24k rows of 768 and 256 columns)
    floatx16 acc[AM], low[AM];
#pragma unroll
    for (int m = 0; m < AM; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = low[m][r] = 0.f;
    uint32_t key[NA];       // the next slab's rows
    Raw8<FT> raw[NA];
    float4 g[NB];
    auto row_a = [&](int i) { return (tid + NT * i) / (TM / 8); };
    auto keys = [&](int slab) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NA; ++i) key[i] = a.uniq_key[min(ub + 32 * slab + row_a(i), ue - 1)];
    };
    auto load = [&](int slab) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
            load_raw8<FT>(raw[i], a.feat_base + (int64_t)key[i] * a.pitch, f0 + (tid + NT * i) % (TM / 8) * 8,
                          ub + 32 * slab + row_a(i) < ue ? a.Fp : 0);
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int x = tid + NT * i, u = ub + 32 * slab + x / (TN / 4), k = n0 + x % (TN / 4) * 4;
            g[i] = k < a.Dp ? *reinterpret_cast<const float4*>(grad + (size_t)min(u, ue - 1) * a.Dp + k) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto stage = [&](int slab) __attribute__((always_inline)) {
        char* const to = smem + (slab & 1) * kStage;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int row = row_a(i), chunk = (tid + NT * i) % (TM / 8);
            if (NT * NA != 32 * TM / 8 && row >= 32) continue;
            uint4 piece[PA];
            split_raw8<FT>(raw[i], piece);
#pragma unroll
            for (int q = 0; q < PA; ++q)
                *reinterpret_cast<uint4*>(to + q * (32 * TM * 2) + row * (2 * TM) + (chunk ^ ((row & TA::kKey) << 2)) * 16) = piece[q];
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int x = tid + NT * i, row = x / (TN / 4), c4 = x % (TN / 4);
            uint2 piece[3];
            split4_bf16(as_x4(g[i]), piece);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<uint2*>(to + kA + q * (32 * TN * 2) + row * (2 * TN) + ((c4 >> 1) ^ ((row & TB::kKey) << 2)) * 16 +
                                          (c4 & 1) * 8) = piece[q];
        }
    };
    // Of a SIMD's two waves (w and w + 4) one splits the next slab while the other multiplies this one, then the
    // other way round: 24k rows of 768 float16 features, 256 columns: 59.5 -> 55 us (waves paired in another way:
    // 57).  The products alone take 37 us, the splitting alone 28.  (float32 features: no registers for a second copy of the code.)
    const bool first = NW < 8 || FT == ET_F32 || wave < 4;
    if (n_slab > 0) {
        keys(0);
        load(0);
        keys(1);
        stage(0);
        load(min(1, n_slab - 1));
        keys(2);
    }
    for (int slab = 0; slab < n_slab; ++slab) {
        __syncthreads();
        auto advance = [&]() __attribute__((always_inline)) {
            stage(slab + 1);
            load(slab + 2);  // (past the end: the last row again, its features as zeros)
            keys(slab + 3);
        };
        if (first && slab + 1 < n_slab) advance();
        const char* ta = smem + (slab & 1) * kStage;
        const char* tb = ta + kA;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            floatx4 fa[AM][PA], fb[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) fb[q] = TB::fragment(tb, q, 32 * wave, ks, lane);
#pragma unroll
            for (int m = 0; m < AM; ++m)
#pragma unroll
                for (int q = 0; q < PA; ++q) fa[m][q] = TA::fragment(ta, q, 32 * m, ks, lane);
            feature_products<PA, AM>(fa, fb, acc, low);
        }
        if (!first && slab + 1 < n_slab) advance();
    }
    const int k = n0 + 32 * wave + (lane & 31);
    if (k >= a.Dp) return;
    float* const out = part + (size_t)split * a.Fp * a.Dp;
#pragma unroll
    for (int m = 0; m < AM; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int f = f0 + 32 * m + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            if (f < a.Fp) out[(size_t)f * a.Dp + k] = acc[m][r] + low[m][r];
        }
}

// float32 rows -> piece matrix
__global__ __launch_bounds__(256) void k_split_matrix(const float* __restrict__ in, int rows, int Dp, int Kp, char* __restrict__ out) {
    const int per_row = Kp / 4, i = blockIdx.x * 256 + threadIdx.x, row = i / per_row, k = (i - row * per_row) * 4;
    if (row >= rows) return;
    store_pieces4(out + (size_t)row * Kp * 6, k, k < Dp ? *reinterpret_cast<const float4*>(in + (size_t)row * Dp + k) : make_float4(0.f, 0.f, 0.f, 0.f));
}
void launch_split_matrix(const float* in, int rows, int Dp, int Kp, void* out, hipStream_t stream) {
    if (rows == 0) return;
    hipLaunchKernelGGL(k_split_matrix, dim3((unsigned)(((int64_t)rows * (Kp / 4) + 255) / 256)), dim3(256), 0, stream, in, rows, Dp, Kp, (char*)out);
}

// columns per workgroup: the whole width up to 256
static int feature_waves(int Dp) { return Dp > 128 ? 8 : Dp > 64 ? 4 : 2; }

void launch_feature_fwd(const FeatureArgs& a, float* hidden, hipStream_t stream) {
    const int nw = feature_waves(a.Dp), gx = (a.Dp + 32 * nw - 1) / (32 * nw), w_pitch = (a.Dp + 31) / 32 * 192;
    // A workgroup of eight waves fills a CU whatever its height, so the kernel chooses it for the rows that it finds: 24k
    // distinct ones of 32k contributions, 768 float16 features and 256 columns take 61 us in tiles of 128, which 32k
    // rows would get, and 56 in tiles of 96, one for every CU.  The grid holds the most workgroups that any number of
    // rows up to max_rows needs: that one, or one of those behind which a height takes another round.  Smaller
    // workgroups share a CU by their LDS: theirs is the height for max_rows.
    // Where the least height gives every CU one tile at most there is nothing to choose (4096 rows of 64 float32
    // features, 256 columns: 7.0 us with the choice, 6.5 without).
    const uint32_t slots = 256 * (8 / nw), rows = a.max_rows;
    int am = feature_tile(rows, gx, slots);
    uint32_t most = feature_tiles(rows, am, gx);
    if (nw == 8 && feature_tiles(rows, 1, gx) > slots) {
        for (int t = 1; t <= 4; ++t)
            for (uint32_t round = 1, r; (r = round * slots / gx * (32 * t)) < rows; ++round)
                most = std::max(most, feature_tiles(r, feature_tile(r, gx, slots), gx));
        am = 0;
    }
    const dim3 grid(most);
#define KGE_FF(F_, A_, W_) hipLaunchKernelGGL((k_feature_fwd<F_, A_, W_>), grid, dim3(W_ * 64), 0, stream, a, (const char*)a.wp, w_pitch, hidden)
#define KGE_FF_A(F_, W_)                                                                             \
    do {                                                                                             \
        if (am == 1) KGE_FF(F_, 1, W_); else if (am == 2) KGE_FF(F_, 2, W_);                         \
        else if (am == 3) KGE_FF(F_, 3, W_); else KGE_FF(F_, 4, W_);                                 \
    } while (0)
#define KGE_FF_W(F_) do { if (nw == 8 && am) KGE_FF(F_, 1, 8); else if (nw == 8) KGE_FF(F_, 0, 8); else if (nw == 4) KGE_FF_A(F_, 4); else KGE_FF_A(F_, 2); } while (0)
    if (a.feat_etype == ET_F16) KGE_FF_W(ET_F16);
    else if (a.feat_etype == ET_BF16) KGE_FF_W(ET_BF16);
    else KGE_FF_W(ET_F32);
#undef KGE_FF
#undef KGE_FF_A
#undef KGE_FF_W
}

// parts of the split contraction: as many as give every CU a workgroup, none with less than four slabs
int feature_grad_parts(int max_rows, int Fp, int Dp) {
    const int nw = feature_waves(Dp), tiles = ((Fp + 127) / 128) * ((Dp + 32 * nw - 1) / (32 * nw));
    return std::max(1, std::min({256 * (8 / nw) / tiles, max_rows / 128, kFeatureGradParts}));
}
void launch_feature_grad(const FeatureArgs& a, const float* grad_rows, float* part, int n_part, hipStream_t stream) {
    const int nw = feature_waves(a.Dp);
    const dim3 grid((unsigned)(((a.Fp + 127) / 128) * ((a.Dp + 32 * nw - 1) / (32 * nw)) * n_part));
#define KGE_FG(F_, W_) hipLaunchKernelGGL((k_feature_grad<F_, 4, W_>), grid, dim3(W_ * 64), 0, stream, a, grad_rows, n_part, part)
#define KGE_FG_W(F_) do { if (nw == 8) KGE_FG(F_, 8); else if (nw == 4) KGE_FG(F_, 4); else KGE_FG(F_, 2); } while (0)
    if (a.feat_etype == ET_F16) KGE_FG_W(ET_F16);
    else if (a.feat_etype == ET_BF16) KGE_FG_W(ET_BF16);
    else KGE_FG_W(ET_F32);
#undef KGE_FG
#undef KGE_FG_W
}

}  // namespace kge
