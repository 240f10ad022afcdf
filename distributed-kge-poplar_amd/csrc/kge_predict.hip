// gfx950 kernel of the prediction sweep's scores (L2 and dot): a few queries against very many table
// rows (src/poplar_kge.cpp:743-808).
//
// Every table row is read once, where it lies and in its own type, and split once into its two scaled float16
// halves (kge_split.h); up to 128 queries meet it, whose halves stay in registers for the whole launch.  Four waves hold
// 32 queries each (128 registers at 256 columns) and multiply a tile of 32 rows (three instructions per
// sixteen columns); four more fetch, four tiles ahead, and split the next tile
// into the other LDS copy.  Waves that do both, one to a SIMD, paid for every instruction's latency
// alone and left the merge kernel beside them no issue slots: 1M float32 rows of 256 columns for 128 queries
// 0.90 ms.  With one tile ahead instead of four a launch of 262144 rows took 174 us, not 130.
// The training forward's kernel, which this replaces for sweeps, splits the 128 queries again for
// every 64 rows, needs 16-bit rows copied to float32 first and takes widths that are no multiple of 64 on
// float32 instructions.  Per pass, before and now, 128 queries: 1M x 256 float32 758 -> 701 us; 500k x 256
// float16 659 -> 503; 300k x 100 float32 459 -> 429; four shards of 100k x 130, 512 queries, 5193 -> 4427;
// 500k x 128, 16 queries, dot: 282 -> 239.
// Three products of halves instead of six of bfloat16 pieces, fragments two steps ahead of their use instead of one, and a tile
// without a cancelled pair stored without a look at its pairs one by one: a launch of 262144 rows beside a merge 154 -> 112 us,
// the pass over 1M x 256 float32 704 -> 644.
// What bounds it: rows (268 MB a launch) and scores (134 MB written here, read by the merge beside it) come to 4.8 TB/s, and a
// workgroup's products, 26 us of the 112, stand between its barriers with its epilogues.
//
#include "kge_loss.h"
#include "kge_split.h"

#include <algorithm>
#include <cstdint>

namespace kge {

struct PredictArgs {
    const float* a;        // queries' predicted tails [n_query, Dp]
    RowSource b;           // rows (no index)
    float* scores;         // [n_query, ldc]
    int n_query, n_row, ldc, Dp;
    int distance_value;    // score = the distance (or the product) itself, else gamma - it
    float gamma;
};

constexpr int PT_ROWS = 32, PT_WAVES = 4;

// four columns of a row, as they lie
template <int ET> struct Raw4 { uint2 v[ET == ET_F32 ? 2 : 1]; };
template <int ET>
DEVINL float4 raw4_f32(const Raw4<ET>& r) {
    if constexpr (ET == ET_F32)
        return make_float4(__uint_as_float(r.v[0].x), __uint_as_float(r.v[0].y), __uint_as_float(r.v[1].x), __uint_as_float(r.v[1].y));
    else
        return load4(reinterpret_cast<const char*>(r.v), 0, ET);
}

// Dot products below this, of rows whose largest elements are 2^14, are computed directly: the elements below 2^-28 of their
// row's largest are off by 2^-50 of it, and where the large ones meet only such ones, they are the product.  (Of ordinary rows'
// one in 10^6 is.)  Rows of zeros have a scale of 0, and no such product.
constexpr float kLeastProduct = 0x1p10f;

template <int DIST, int ET, int NS>  // ET: the rows' element type, NS: slabs of 32 columns
__global__ __launch_bounds__(2 * PT_WAVES * 64, 1) void k_predict_scores(PredictArgs p) {
    using Tile = RowTile<PT_ROWS, 2>;
    constexpr int PF = 4;                    // tiles asked for ahead (even: a register set stays with its LDS copy)
    constexpr int kBuf = NS * Tile::kBytes;
    __shared__ __attribute__((aligned(16))) char smem[2 * kBuf];
    __shared__ float na_s[32 * PT_WAVES], sa_s[32 * PT_WAVES], nb_s[2][PT_ROWS], sb_s[2][PT_ROWS];  // squared norms and scales
    // tid: within the four waves of this role
    const int tid = threadIdx.x & (PT_WAVES * 64 - 1), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int Dp = p.Dp, n_tile = (p.n_row + PT_ROWS - 1) / PT_ROWS;
    const int step = gridDim.x;
    int tile = blockIdx.x;
    if (tile >= n_tile) return;

    if (threadIdx.x >= PT_WAVES * 64) {
        // waves 4 .. 7: rows into halves.  Thread -> row, four columns of every slab.
        const int s_row = tid >> 3, c4 = tid & 7;
        char* const s_at = smem + s_row * 64 + ((c4 >> 1) ^ ((s_row >> 2) & 3)) * 16 + (c4 & 1) * 8;
        Raw4<ET> raw[PF][NS];
        auto fetch = [&](Raw4<ET> (&raw)[NS], int t) __attribute__((always_inline)) {  // past the last row or tile: the last again
            const char* const row = p.b.base + (int64_t)min(t * PT_ROWS + s_row, p.n_row - 1) * p.b.pitch;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                int k = 32 * s + 4 * c4;
                if (s >= NS - 2) k = min(k, Dp - 4);  // only the last two slabs may reach past Dp (zeros when staged)
                const char* at = row + (size_t)k * (ET == ET_F32 ? 4 : 2);
                if constexpr (ET == ET_F32) {
                    const uint4 t4 = *reinterpret_cast<const uint4*>(at);
                    raw[s].v[0] = make_uint2(t4.x, t4.y); raw[s].v[1] = make_uint2(t4.z, t4.w);
                } else {
                    raw[s].v[0] = *reinterpret_cast<const uint2*>(at);
                }
            }
        };
        static_for<PF>([&](auto x) __attribute__((always_inline)) { fetch(raw[x.value], min(tile + x.value * step, n_tile - 1)); });
        while (tile < n_tile)
            static_for<PF>([&](auto x) __attribute__((always_inline)) {
                if (tile >= n_tile) return;
                constexpr int buf = x.value & 1;
                float sq = 0.f, top = 0.f;
                auto value = [&](int s) __attribute__((always_inline)) {
                    const float4 v = raw4_f32<ET>(raw[x.value][s]);
                    return s >= NS - 2 && 32 * s + 4 * c4 >= Dp ? make_float4(0.f, 0.f, 0.f, 0.f) : v;
                };
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const float4 v = value(s);
                    if (DIST == DIST_L2) sq += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
                    top = fmaxf(fmaxf(top, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
                }
                // (a row's eight threads)
                top = fmaxf(top, swap1(top));
                top = fmaxf(top, swap2(top));
                top = fmaxf(top, mirror8(top));
                const float scale = half_scale(top), up = pow2_inverse(scale);
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const float4 v = value(s);
                    uint32_t lo[2], hi[2];
                    split2_f16(v.x * up, v.y * up, lo);
                    split2_f16(v.z * up, v.w * up, hi);
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        *reinterpret_cast<uint2*>(s_at + buf * kBuf + s * Tile::kBytes + q * (PT_ROWS * 64)) = make_uint2(lo[q], hi[q]);
                }
                fetch(raw[x.value], min(tile + PF * step, n_tile - 1));
                if (DIST == DIST_L2) {
                    sq += swap1(sq);
                    sq += swap2(sq);
                    sq += mirror8(sq);
                }
                if (c4 == 0) {
                    nb_s[buf][s_row] = sq;
                    sb_s[buf][s_row] = DIST == DIST_L2 || top != 0.f ? scale : 0.f;  // (dot: the products of zeros are right)
                }
                // barrier i: tile i is in LDS; the other waves then multiply it while tile i + 1 is staged into
                // the copy that they left before barrier i
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                tile += step;
            });
        return;
    }

    // waves 0 .. 3: 32 queries each (a wave without any keeps the barriers).  Lane's query q0 + lane % 32,
    // columns 16 ks + 8 (lane / 32) .. + 7 of step ks.
    const int q0 = blockIdx.y * (32 * PT_WAVES) + 32 * wave;
    const bool active = q0 < p.n_query;
    floatx4 fa[2 * NS][2];
    float na = 0.f, top = 0.f;
    auto query4 = [&](int ks, int h) __attribute__((always_inline)) {
        const int k = 16 * ks + 8 * (lane >> 5) + 4 * h;
        const float4 v = *reinterpret_cast<const float4*>(p.a + (size_t)min(q0 + (lane & 31), p.n_query - 1) * Dp + min(k, Dp - 4));
        return k >= Dp ? make_float4(0.f, 0.f, 0.f, 0.f) : v;
    };
#pragma unroll
    for (int ks = 0; ks < 2 * NS; ++ks)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4 v = query4(ks, h);
            na += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
            top = fmaxf(fmaxf(top, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
        }
    na += __shfl_xor(na, 32, 64);
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    const float scale_a = half_scale(top), up_a = pow2_inverse(scale_a);
    if (lane < 32) {  // (read by this wave alone)
        na_s[32 * wave + lane] = na;
        sa_s[32 * wave + lane] = DIST == DIST_L2 ? -2.f * scale_a : top != 0.f ? scale_a : 0.f;
    }
    asm volatile("" ::: "memory");  // (the rows are read again, not kept)
#pragma unroll
    for (int ks = 0; ks < 2 * NS; ++ks) {
        uint32_t w[2][2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4 v = query4(ks, h);
            split2_f16(v.x * up_a, v.y * up_a, w[h][0]);
            split2_f16(v.z * up_a, v.w * up_a, w[h][1]);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
            fa[ks][q] = __builtin_bit_cast(floatx4, uint4{w[0][0][q], w[0][1][q], w[1][0][q], w[1][1][q]});
    }
    for (int buf = 0; tile < n_tile; tile += step, buf ^= 1) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (!active) continue;
        const char* const cur = smem + buf * kBuf;
        floatx16 big, small[2];  // in turn: an instruction does not wait for the one before it
#pragma unroll
        for (int r = 0; r < 16; ++r) big[r] = small[0][r] = small[1][r] = 0.f;
        // this step's fragments and the next ones': a step's products are done before a read of its time is back
        constexpr int kAhead = 2;
        floatx4 fb[kAhead + 1][2];
        auto read = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < 2; ++q) fb[ks % (kAhead + 1)][q] = Tile::fragment(cur + ks / 2 * Tile::kBytes, q, 0, ks & 1, lane);
        };
#pragma unroll
        for (int ks = 0; ks < kAhead; ++ks) read(ks);
#pragma unroll
        for (int ks = 0; ks < 2 * NS; ++ks) {
            if (ks + kAhead < 2 * NS) read(ks + kAhead);
            auto product = [&](int qa, int qb, floatx16 acc) __attribute__((always_inline)) {
                return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fa[ks][qa]),
                                                              __builtin_bit_cast(f16x8, fb[ks % (kAhead + 1)][qb]), acc, 0, 0, 0);
            };
            small[0] = product(0, 1, small[0]);
            small[1] = product(1, 0, small[1]);
            big = product(0, 0, big);
            __builtin_amdgcn_sched_barrier(0);  // the reads stay a step ahead of their use
        }

        // register r of lane l: query 8 (r / 4) + 4 (l / 32) + r % 4, row l % 32
        const int n = tile * PT_ROWS + (lane & 31), hl = lane >> 5;
        const float nb = DIST == DIST_L2 ? nb_s[buf][lane & 31] : 0.f, sb = sb_s[buf][lane & 31];
        auto put = [&](int q, int row, float v) __attribute__((always_inline)) {
            const float dist = DIST == DIST_L2 ? __builtin_amdgcn_sqrtf(v) : v;  // (never negative; a NaN stays one)
            p.scores[(size_t)q * p.ldc + row] = p.distance_value ? dist : p.gamma - dist;
        };
        float val[16];
        uint64_t bad = 0u;
        float least = INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = 8 * (r >> 2) + 4 * hl + (r & 3);
            const float product = fmaf(small[0][r] + small[1][r], kHalfStep, big[r]), scale = sa_s[32 * wave + m];
            if (DIST == DIST_L2) {
                const float ns = na_s[32 * wave + m] + nb;
                val[r] = fmaf(product, scale * sb, ns);
                bad |= __ballot(!(val[r] >= kCancelRatio * ns));
            } else {
                val[r] = product * scale * sb;
                bad |= __ballot(!(fabsf(val[r]) < INFINITY));
                least = fminf(least, fabsf(product));
            }
        }
        if (DIST != DIST_L2) bad |= __ballot(least < kLeastProduct);
        if (!bad && q0 + 32 <= p.n_query && (tile + 1) * PT_ROWS <= p.n_row) {  // the rule: all of them, without a look at any
            float* const out = p.scores + (size_t)q0 * p.ldc + tile * PT_ROWS;
            const uint32_t off = (uint32_t)(4 * hl * p.ldc + (lane & 31));
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float dist = DIST == DIST_L2 ? __builtin_amdgcn_sqrtf(val[r]) : val[r];
                (out + (size_t)(8 * (r >> 2) + (r & 3)) * p.ldc)[off] = p.distance_value ? dist : p.gamma - dist;
            }
            continue;
        }
        if (!bad) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int q = q0 + 8 * (r >> 2) + 4 * hl + (r & 3);
                if (n < p.n_row && q < p.n_query) put(q, n, val[r]);
            }
            continue;
        }
        uint32_t again = 0u;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = 8 * (r >> 2) + 4 * hl + (r & 3);
            const bool good = DIST == DIST_L2 ? val[r] >= kCancelRatio * (na_s[32 * wave + m] + nb)
                                              : fabsf(val[r]) < INFINITY && fabsf(val[r]) >= kLeastProduct * sa_s[32 * wave + m] * sb;
            if (n < p.n_row && q0 + m < p.n_query) {
                if (good) put(q0 + m, n, val[r]); else again |= 1u << r;
            }
        }
        // rare: the wave computes pairs directly, eight at a time, eight lanes to a pair (two pairs of each
        // of four lanes; fewer lanes: the last one's again): those that cancelled, the smallest products, and those that are not
        // finite (an infinity's halves are infinity and NaN; from the values themselves its distance is
        // infinite and its row comes last, a NaN's score is NaN and the merge takes none).  Each round is a
        // ballot, a shuffle and trips to L2, one after the other, which four waves to a CU do not hide: at two
        // pairs a round, through shuffles back to the lanes whose registers they were, a table whose rows lie
        // close together (every pair cancelled; 200k x 256 float32, 128 queries) took 12.4 ms.
        uint64_t owners;
        while ((owners = __ballot(again != 0u)) != 0) {
            int own[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                own[i] = owners ? __ffsll((long long)owners) - 1 : own[i ? i - 1 : 0];
                owners &= owners - 1;
            }
            const int src = lane & 32 ? (lane & 16 ? own[3] : own[2]) : (lane & 16 ? own[1] : own[0]);
            const uint32_t bits = __shfl(again, src, 64), upper = bits & (bits - 1);
            const int fr = __ffs((int)((lane & 8) && upper ? upper : bits)) - 1;
            const int q = q0 + 8 * (fr >> 2) + 4 * (src >> 5) + (fr & 3), row = tile * PT_ROWS + (src & 31);
            const float* ar = p.a + (size_t)q * Dp;
            const char* br = p.b.base + (int64_t)row * p.b.pitch;
            float part = 0.f;
#pragma unroll 1
            for (int k0 = 4 * (lane & 7); k0 < Dp; k0 += 128) {
                float4 x[4], y[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {  // four loads of each row under way
                    const int k = k0 + 32 * i;
                    x[i] = y[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (k < Dp) { x[i] = *reinterpret_cast<const float4*>(ar + k); y[i] = load4(br, k, ET); }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (DIST == DIST_L2) {
                        const float dx = x[i].x - y[i].x, dy = x[i].y - y[i].y, dz = x[i].z - y[i].z, dw = x[i].w - y[i].w;
                        part += dx * dx + dy * dy + dz * dz + dw * dw;
                    } else {
                        part += x[i].x * y[i].x + x[i].y * y[i].y + x[i].z * y[i].z + x[i].w * y[i].w;
                    }
                }
            }
#pragma unroll
            for (int o = 4; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
            if ((lane & 7) == 0) put(q, row, part);
            if (lane == own[0] || lane == own[1] || lane == own[2] || lane == own[3]) {
                again &= again - 1;
                again &= again - 1;
            }
        }
    }
}

// Whether launch_predict_scores takes a sweep.  Up to 256 columns, as many as the registers hold the
// queries of; L2 and dot only (L1 has no product form), by halves only.
bool predict_scores_takes(const ScoreShape& sh) {
    if (sh.use_mfma != 2 || sh.score_fn == SCORE_TRANSH || sh.Dp > 256) return false;
    return sh.score_fn == SCORE_DISTMULT || sh.dist_fn != DIST_L1;
}

// scores[q * ldc + r] of queries a [sh.B, Dp] against rows 0 .. n_row - 1 of `b` (16-byte aligned sections)
void launch_predict_scores(const ScoreShape& sh, const float* a, const RowSource& b, int n_row, float* scores, int ldc,
                           hipStream_t stream) {
    PredictArgs p = {a, b, scores, sh.B, n_row, ldc, sh.Dp, score_is_distance_value(sh.score_fn) ? 1 : 0, sh.gamma};
    const bool l2 = sh.score_fn != SCORE_DISTMULT && sh.dist_fn == DIST_L2;
    // A workgroup fills its CU and stays for the launch, so the merge of the chunk before (a workgroup per
    // query, two to a CU) needs CUs of its own beside it: 1M rows for 128 queries on all 256 CUs 0.90 ms,
    // on 192 0.73.  What is left is divided among the groups of 128 queries, whose workgroups walk the
    // same tiles at the same time.
    const int groups = (sh.B + 32 * PT_WAVES - 1) / (32 * PT_WAVES), cus = 256 - std::min(64, (sh.B + 1) / 2);
    const dim3 grid((unsigned)std::min(std::max(1, cus / groups), (n_row + PT_ROWS - 1) / PT_ROWS), (unsigned)groups);
#define KGE_PS(D_, E_, N_) hipLaunchKernelGGL((k_predict_scores<D_, E_, N_>), grid, dim3(2 * PT_WAVES * 64), 0, stream, p)
#define KGE_PS_N(D_, E_)                                                                    \
    do {                                                                                    \
        if (sh.Dp <= 64) KGE_PS(D_, E_, 2); else if (sh.Dp <= 128) KGE_PS(D_, E_, 4);       \
        else if (sh.Dp <= 192) KGE_PS(D_, E_, 6); else KGE_PS(D_, E_, 8);                   \
    } while (0)
#define KGE_PS_E(D_)                                                                        \
    do {                                                                                    \
        if (b.etype == ET_F32) KGE_PS_N(D_, ET_F32);                                        \
        else if (b.etype == ET_BF16) KGE_PS_N(D_, ET_BF16); else KGE_PS_N(D_, ET_F16);      \
    } while (0)
    if (l2) KGE_PS_E(DIST_L2); else KGE_PS_E(DIST_DOT);
#undef KGE_PS
#undef KGE_PS_N
#undef KGE_PS_E
}

}  // namespace kge
