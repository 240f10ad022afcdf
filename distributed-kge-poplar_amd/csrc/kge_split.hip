// gfx950 scoring kernels on three-piece operands (L2 and dot): the operand gather, the forward
// scores with the fused loss, and both sides of the backward.
//
// Every float32 value is the exact sum of three bfloat16 pieces, and a float32 product is six
// products of pieces (split4_bf16, mfma_split6's order).  Splitting while staging, as a kernel
// that reads float32 operands must, costs more vector instructions than the products cost matrix
// instructions, and every tile that reads a row splits it again.  Here every value is split once,
// by the kernel that makes it: the gather writes the operand rows as pieces, the forward writes the
// backward's coefficients as pieces, and the product kernels copy tiles straight from memory into
// LDS (global_load_lds, no registers, no vector instructions), so that their waves do little else
// than read fragments and multiply.
//
#include "kge_device.h"
#include "kge_loss.h"
#include "kge_split.h"

#include <algorithm>
#include <cstdint>

namespace kge {

// --------------------------------------------------------------------------
// operand gather: RPW contributions per wave, their entity (or hidden) rows with the relation
// applied for the heads, as pieces; and the rows' squared norms.
template <int RPW, bool XF>  // XF: the complex product and the rotation compiled in
__global__ __launch_bounds__(256) void k_gather_pieces(RowSource ent, const float* __restrict__ rel,
                                                       const uint32_t* __restrict__ crel, int rel_mode, int half,
                                                       int n_head, int n_rows, int Dp, int Kp, char* __restrict__ out,
                                                       float* __restrict__ norm, TailCols tc) {
    const int lane = threadIdx.x & 63;
    const int c0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW;
    if (c0 >= n_rows) return;
    // the row numbers are asked for together with the block's tail count (rows past it are
    // never used, but their slots hold valid numbers): one round trip instead of two
    uint32_t key[RPW], rkey[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        const int c = min(c0 + r, n_rows - 1);  // a row past the end repeats the last one
        key[r] = ent.index ? ent.index[c] : (uint32_t)c;
        rkey[r] = (c < n_head && rel_mode) ? crel[c] : 0u;
    }
    bool live[RPW], any = false;
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        live[r] = c0 + r < n_rows && tc.live(c0 + r - n_head);
        any = any || live[r];
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r) asm volatile("" : "+v"(key[r]), "+v"(rkey[r]));
    if (!any) return;
    const char* row[RPW];
    const float* rrow[RPW];
    float sq[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        row[r] = ent.base + (int64_t)key[r] * ent.pitch;
        rrow[r] = (c0 + r < n_head && rel_mode) ? rel + (size_t)rkey[r] * Dp : nullptr;
        sq[r] = 0.f;
    }
    for (int k = lane * 4; k < Kp; k += 256) {
        float4 v[RPW], w[RPW];
#pragma unroll
        for (int r = 0; r < RPW; ++r) {  // all loads first
            v[r] = w[r] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (k < Dp) {
                v[r] = load4(row[r], k, ent);
                if (rrow[r] && rel_mode <= 2) w[r] = *reinterpret_cast<const float4*>(rrow[r] + k);
            }
        }
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            if (rrow[r] && k < Dp) {
                if (XF && rel_mode >= 3) v[r] = relation_xf(v[r], row[r], ent.etype, rrow[r], k, half, rel_mode);
                else v[r] = rel_mode == 1 ? f4add(v[r], w[r]) : f4mul(v[r], w[r]);
            }
            sq[r] += v[r].x * v[r].x + v[r].y * v[r].y + v[r].z * v[r].z + v[r].w * v[r].w;
            if (live[r]) store_pieces4(out + (size_t)(c0 + r) * Kp * 6, k, v[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        const float s = wave_sum(sq[r]);
        if (lane == 0 && live[r]) norm[c0 + r] = s;
    }
}

void launch_gather_pieces(const RowSource& ent, const float* rel, const uint32_t* crel, int rel_mode, int half,
                          int n_head, int n_rows, int Dp, int Kp, void* out, float* norm, hipStream_t stream,
                          const TailCols* tail_cols) {
    TailCols tc = {};
    if (tail_cols) tc = *tail_cols;
    // two rows per wave where that leaves enough waves: the kernel is resident waves over the
    // latency of the chain row number -> row -> store, and a wave may as well keep two chains going
#define KGE_GATHER(N_, X_)                                                                                            \
    hipLaunchKernelGGL((k_gather_pieces<N_, X_>), dim3((n_rows + 4 * N_ - 1) / (4 * N_)), dim3(256), 0, stream, ent, rel, \
                       crel, rel_mode, half, n_head, n_rows, Dp, Kp, (char*)out, norm, tc)
    if (rel_mode >= 3) KGE_GATHER(1, true);
    else if (n_rows >= 8192) KGE_GATHER(2, false);
    else KGE_GATHER(1, false);
#undef KGE_GATHER
}

// --------------------------------------------------------------------------
// products

// Tiles of 64 x 64, four waves, three workgroups to a CU: at these sizes a launch is bound by the
// latency of its slabs and by how many workgroups there are, not by the matrix cores.
constexpr int kTile = 64, kWaves = 2;  // waves as kWaves x kWaves

// The product loop of a TM x TN tile: n_slab slabs of 32 contraction steps, two tile copies in LDS
// (one fills while the other is multiplied, one barrier per slab).  TA, TB: RowTile / ColTile;
// a_step, b_step: bytes from slab to slab.  Waves as WM x WN, each (TM/WM) x (TN/WN) in 32 x 32
// accumulators.
// b_rows: rows of `b` along the contraction where it lies across it (ColTile).  The last slab's rows past them
// repeat the last one: their coefficients are zero, but what lies behind a block's rows are other
// blocks', and zero times a neighbour's infinity or NaN would be this block's NaN.
template <class TA, class TB, int TM, int TN, int WM, int WN>
struct SplitProduct {
    static constexpr int NW = WM * WN, AM = TM / WM / 32, AN = TN / WN / 32;
    static constexpr int kStage = TA::kBytes + TB::kBytes, kLds = 2 * kStage;
    static constexpr int kCopies = TA::kCopies + TB::kCopies, kEach = kCopies / NW;
    static_assert(kCopies % NW == 0, "every wave issues the same number of copies");

    // meanwhile(): what the caller has to fetch for itself, under the first slab's way from memory
    template <class Meanwhile>
    static DEVINL void run(char* smem, const char* a, int a_pitch, size_t a_step, const char* b, int b_pitch, size_t b_step,
                           int n_slab, int b_rows, floatx16 (&acc)[AM][AN], int lane, int wave, Meanwhile&& meanwhile) {
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
            const uint32_t to = lds0 + (slab & 1) * kStage;
            if constexpr (!std::is_same_v<TB, RowTile<TN>>) {
                const int last = b_rows - 32 * slab - 1;
                if (last < 31)  // the last slab's offsets take the others' place
#pragma unroll
                    for (int i = 0; i < kEach; ++i) {
                        const int x = wave + NW * i;
                        if (x >= TA::kCopies) off[i] = TB::source(x - TA::kCopies, lane, b_pitch, last);
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
        const int wm = (wave / WN) * (TM / WM), wn = (wave % WN) * (TN / WN);
        for (int slab = 0; slab < n_slab; ++slab) {
            wait_copies_and_barrier<0>();
            if (slab + 1 < n_slab) fill(slab + 1);
            const char* ta = smem + (slab & 1) * kStage;
            const char* tb = ta + TA::kBytes;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                floatx4 fa[AM][3], fb[AN][3];
#pragma unroll
                for (int q = 0; q < 3; ++q) {
#pragma unroll
                    for (int m = 0; m < AM; ++m) fa[m][q] = TA::fragment(ta, q, wm + 32 * m, ks, lane);
#pragma unroll
                    for (int n = 0; n < AN; ++n) fb[n][q] = TB::fragment(tb, q, wn + 32 * n, ks, lane);
                }
                // six products, smallest first; the accumulators in turn, so that an instruction
                // does not wait for the one before it
                constexpr int qa[6] = {0, 2, 1, 0, 1, 0}, qb[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
                for (int x = 0; x < 6; ++x)
#pragma unroll
                    for (int m = 0; m < AM; ++m)
#pragma unroll
                        for (int n = 0; n < AN; ++n)
                            acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                __builtin_bit_cast(bf16x8, fa[m][qa[x]]), __builtin_bit_cast(bf16x8, fb[n][qb[x]]),
                                acc[m][n], 0, 0, 0);
            }
        }
    }
};

// --------------------------------------------------------------------------
// the coefficient matrix as pieces

// A 32 x 32 block of coefficients in accumulator layout (register r of lane l: row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32) to its place in the piece matrix, block corner
// (m0, n0) of block d.  Neighbouring lanes swap values so that a lane stores two columns of one row as
// one word.  For L2 also the block's row sums and column sums.
template <int DIST>
DEVINL void store_coef_block(const float (&c)[16], const SplitCoef& p, int d, int m0, int n0, int lane) {
    const int Bp = p.Bp, Tp = p.Tp;
    if (m0 >= Bp || n0 >= Tp) return;
    const int cl = lane & 31, hl = lane >> 5;
    const bool odd = lane & 1, b1 = lane & 2, b2 = lane & 4, b3 = lane & 8;
    char* const base = p.coefp + ((size_t)d * Bp + m0) * Tp * 6 + (size_t)(n0 >> 5) * 192 + (cl & ~1) * 2;
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float got = swap1(odd ? c[2 * i] : c[2 * i + 1]);
        const float x = odd ? got : c[2 * i], y = odd ? c[2 * i + 1] : got;  // row 2 i + odd of this lane's half
        s[i] = x + y;
        uint32_t w[3];
        split2(x, y, w);
        char* const q = base + (size_t)(8 * (i >> 1) + 4 * hl + 2 * (i & 1) + odd) * Tp * 6;
#pragma unroll
        for (int k = 0; k < 3; ++k) *reinterpret_cast<uint32_t*>(q + 64 * k) = w[k];
    }
    if (DIST != DIST_L2) return;
    // row sums: at each step a lane keeps half of its rows and hands the other half's sums over
    float t[4], u[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = (b1 ? s[2 * i + 1] : s[2 * i]) + swap2(b1 ? s[2 * i] : s[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < 2; ++i) u[i] = (b2 ? t[2 * i + 1] : t[2 * i]) + __shfl_xor(b2 ? t[2 * i] : t[2 * i + 1], 4, 64);
    float v = (b3 ? u[1] : u[0]) + __shfl_xor(b3 ? u[0] : u[1], 8, 64);
    v += __shfl_xor(v, 16, 64);
    const int r = lane & 15;
    if (!(lane & 16))
        p.rowpart[((size_t)d * Bp + m0 + 8 * (r >> 2) + 4 * hl + (r & 3)) * (Tp >> 5) + (n0 >> 5)] = v;
    float col = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) col += c[k];
    col += __shfl_xor(col, 32, 64);
    if (lane < 32) p.colpart[((size_t)d * (Bp >> 5) + (m0 >> 5)) * Tp + n0 + lane] = col;
}

// The same from float32 coefficients in memory (the losses that are formed row by row): one wave
// per 32 x 32 block.
template <int DIST>
__global__ __launch_bounds__(256) void k_coef_pieces(ScoreShape sh, const float* __restrict__ coef,
                                                     const uint32_t* __restrict__ nearflag, SplitCoef p) {
    const int lane = threadIdx.x & 63, MT = p.Bp >> 5, NT = p.Tp >> 5;
    const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int d = g / (MT * NT), mt = (g - d * MT * NT) / NT, nt = g % NT;
    if (d >= sh.S || 32 * nt >= tail_limit(sh.tcount, d, sh.T, sh.tpad)) return;
    const float* src = coef + (size_t)d * sh.B * sh.T;
    const bool skip = DIST == DIST_L2 && nearflag[((size_t)d * MT + mt) * NT + nt] != 0u;  // direct form
    const int n = 32 * nt + (lane & 31);
    float c[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = 32 * mt + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        c[r] = (!skip && m < sh.B && n < sh.T) ? src[(size_t)m * sh.T + n] : 0.f;
    }
    store_coef_block<DIST>(c, p, d, 32 * mt, 32 * nt, lane);
}

// --------------------------------------------------------------------------
// forward

// (kCancelRatio, kNearRatio: kge_loss.h)
template <int DIST, int OM>
__global__ __launch_bounds__(kWaves * kWaves * 64, 2) void k_split_fwd(SplitFwd p) {
    constexpr int TM = kTile, TN = kTile, WM = kWaves, WN = kWaves;
    using P = SplitProduct<RowTile<TM>, RowTile<TN>, TM, TN, WM, WN>;
    __shared__ __attribute__((aligned(16))) char smem[P::kLds];
    __shared__ float na_s[TM], nb_s[TN], mult_s[TN], red[WM * WN];
    __shared__ uint32_t label_s[TM];
    const ScoreShape& sh = p.sh;
    const int B = sh.B, T = sh.T, Kp = p.Kp;
    const TileId tile = xcd_tile((T + TN - 1) / TN, (B + TM - 1) / TM, sh.S);
    const int d = tile.z, m0 = tile.y * TM, n0 = tile.x * TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t_live = tail_limit(sh.tcount, d, T, sh.tpad);
    if (n0 >= t_live) {  // merged tails: the block has no such column
        if (OM == 0 && tid == 0) p.loss_part[(size_t)d * (tile.gx * tile.gy) + tile.y * tile.gx + tile.x] = 0.f;
        return;
    }
    const int n_live = sh.tcount ? (int)sh.tcount[d] : T;
    const int a_row = d * B, b_row = p.b_c0 + d * T;
    const int pitch = Kp * 6;
    const char* a = p.rows + (int64_t)(a_row + m0) * pitch;
    const char* b = p.rows + (int64_t)(b_row + n0) * pitch;
    floatx16 acc[P::AM][P::AN];
#pragma unroll
    for (int m = 0; m < P::AM; ++m)
#pragma unroll
        for (int n = 0; n < P::AN; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
    P::run(smem, a, pitch, 192, b, pitch, 192, Kp / 32, 0, acc, lane, wave, [&]() __attribute__((always_inline)) {
        for (int i = tid; i < TM; i += WM * WN * 64) {
            if (DIST == DIST_L2) na_s[i] = p.norm[a_row + m0 + i];
            if (OM == 0) label_s[i] = m0 + i < B ? p.clabel[d * B + m0 + i] : 0u;
        }
        if (DIST == DIST_L2)
            for (int i = tid; i < TN; i += WM * WN * 64) nb_s[i] = p.norm[b_row + n0 + i];
        if (OM == 0)
            for (int i = tid; i < TN; i += WM * WN * 64)
                mult_s[i] = n0 + i < T ? (sh.tmult ? sh.tmult[(size_t)d * T + n0 + i] : 1.f) : 0.f;
    });

    // epilogue.  Register r of lane l holds row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
    const int wm = (wave / WN) * (TM / WM), wn = (wave % WN) * (TN / WN);
    const int cl = lane & 31, hl = lane >> 5;
    const float Tn = (float)T;
    const float w_pos = uniform_f32(0.5f * Tn), w_neg = uniform_f32((0.5f * Tn) / (float)(T - 1));
    const float inv_norm = uniform_f32(1.f / ((float)sh.S * (float)B * Tn));
    const float grad_scale = uniform_f32(inv_norm * sh.loss_scale);
    const int Bp = p.out.Bp, Tp = p.out.Tp, MT = Bp >> 5, NT = Tp >> 5;
    float loss_acc = 0.f;
#pragma unroll
    for (int mi = 0; mi < P::AM; ++mi)
#pragma unroll
        for (int ni = 0; ni < P::AN; ++ni) {
            const int mb = wm + 32 * mi, nbk = wn + 32 * ni;  // the sub-block's corner in the tile
            const int n = n0 + nbk + cl;
            // columns behind a block's distinct tails repeat its first row, the most popular one more
            // often than not: no pair of theirs is worth a second look
            const bool col_counts = n < n_live;
            float val[16];
            uint32_t cancel = 0u, near = 0u;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                val[r] = acc[mi][ni][r];
                const int m_loc = mb + 8 * (r >> 2) + 4 * hl + (r & 3);
                const bool live = col_counts && m0 + m_loc < B;
                bool good = fabsf(val[r]) < INFINITY;  // (dot)
                if (DIST == DIST_L2) {
                    const float ns = na_s[m_loc] + nb_s[nbk + cl];
                    val[r] = ns - 2.f * val[r];
                    good = val[r] >= kCancelRatio * ns;
                    if (live && val[r] < kNearRatio * ns) near |= 1u << r;
                }
                if (!good) cancel |= 1u << r;
            }
            // rare: the wave recomputes pairs directly, two pairs of each of two lanes at a time, sixteen
            // lanes to a pair: those that cancelled, and those that are not finite (an infinity's second
            // piece is NaN).  Pairs that do not count, a NaN among them, get any finite value.
            if (__ballot(cancel != 0u)) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (!(col_counts && m0 + mb + 8 * (r >> 2) + 4 * hl + (r & 3) < B)) {
                        val[r] = 0.f;
                        cancel &= ~(1u << r);
                    }
                near = 0u;
                uint32_t left = cancel;
                uint64_t owners;
                while ((owners = __ballot(left != 0u)) != 0) {
                    const int l0 = __ffsll((long long)owners) - 1;
                    const uint64_t rest = owners & (owners - 1);
                    const int l1 = rest ? __ffsll((long long)rest) - 1 : l0;
                    const int src = lane & 32 ? l1 : l0;
                    const uint32_t bits = __shfl(left, src, 64), upper = bits & (bits - 1);
                    const int fr = __ffs((int)((lane & 16) && upper ? upper : bits)) - 1;
                    const char* ar = a + (int64_t)(mb + 8 * (fr >> 2) + 4 * (src >> 5) + (fr & 3)) * pitch;
                    const char* br = b + (int64_t)(nbk + (src & 31)) * pitch;
                    float part = 0.f;
                    for (int k = (lane & 15) * 4; k < Kp; k += 64) {
                        const float4 x = load_pieces4(ar, k), y = load_pieces4(br, k);
                        if (DIST == DIST_L2) {
                            const float dx = x.x - y.x, dy = x.y - y.y, dz = x.z - y.z, dw = x.w - y.w;
                            part += dx * dx + dy * dy + dz * dz + dw * dw;
                        } else {
                            part += x.x * y.x + x.y * y.y + x.z * y.z + x.w * y.w;
                        }
                    }
#pragma unroll
                    for (int o = 8; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
                    const int at = (lane == l0) ? 0 : 32;
                    const float v0 = __shfl(part, at, 64), v1 = __shfl(part, at + 16, 64);
                    if (lane == l0 || lane == l1) {
                        const uint32_t up = left & (left - 1);
                        const uint32_t b0 = left ^ up, b1 = up & (0u - up);
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            if ((b0 >> r) & 1u) val[r] = v0;
                            if ((b1 >> r) & 1u) val[r] = v1;
                        }
                        left = up & (up - 1);
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m_loc = mb + 8 * (r >> 2) + 4 * hl + (r & 3);
                    if (DIST == DIST_L2 && col_counts && m0 + m_loc < B && val[r] < kNearRatio * (na_s[m_loc] + nb_s[nbk + cl]))
                        near |= 1u << r;
                }
            }
            const bool flagged = DIST == DIST_L2 && __ballot(near != 0u) != 0;
            if (DIST == DIST_L2 && p.nearflag && lane == 0 && m0 + mb < Bp && n0 + nbk < Tp)
                p.nearflag[((size_t)d * MT + ((m0 + mb) >> 5)) * NT + ((n0 + nbk) >> 5)] = flagged ? 1u : 0u;
            if (OM != 0) {  // raw scores (and distances)
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
                continue;
            }
            const float mult = mult_s[nbk + cl];
            float c[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m_loc = mb + 8 * (r >> 2) + 4 * hl + (r & 3);
                const bool live = m0 + m_loc < B && n < T;
                const float dist = DIST == DIST_L2 ? __builtin_amdgcn_sqrtf(val[r]) : val[r];  // (never negative; a NaN stays one)
                const float score = score_is_distance_value(sh.score_fn) ? dist : sh.gamma - dist;
                float ds;
                const float term = logsigmoid_column(score, (uint32_t)n == label_s[m_loc], mult, w_pos, w_neg, grad_scale, ds);
                if (live) loss_acc += term;
                float v = score_is_distance_value(sh.score_fn) ? ds : -ds;
                if (DIST == DIST_L2) v = dist != 0.f ? v * __builtin_amdgcn_rcpf(dist) : 0.f;
                c[r] = live ? v : 0.f;
            }
            if (flagged) {  // the backward takes this block in the direct form, from the coefficients as they are
                float* const out = p.coef + (size_t)d * B * T;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + mb + 8 * (r >> 2) + 4 * hl + (r & 3);
                    if (m < B && n < T) out[(size_t)m * T + n] = c[r];
                    c[r] = 0.f;
                }
            }
            store_coef_block<DIST>(c, p.out, d, m0 + mb, n0 + nbk, lane);
        }
    if (OM == 0) {
        loss_acc = wave_sum(loss_acc);
        if (lane == 0) red[wave] = loss_acc;
        __syncthreads();
        if (tid == 0) {
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

template <int DIST, bool SIDE_B>
DEVINL void split_bwd_tile(const SplitBwd& p, int d, int tile_x, int tile_y, char* smem, float* csum_s) {
    constexpr int TM = kTile, TN = kTile, WM = kWaves, WN = kWaves;
    using TA = std::conditional_t<SIDE_B, ColTile<TM>, RowTile<TM>>;
    using P = SplitProduct<TA, ColTile<TN>, TM, TN, WM, WN>;
    const int i0 = tile_y * TM, kt0 = tile_x * TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int B = p.B, T = p.T, Bp = p.in.Bp, Tp = p.in.Tp, MT = Bp >> 5, NT = Tp >> 5, pitch = p.Kp * 6;
    const int t_live = tail_limit(p.tcount, d, T, p.tpad);  // merged tails: the block's live columns
    const int n_self = SIDE_B ? t_live : B, n_other = SIDE_B ? B : t_live, n_slab = (n_other + 31) >> 5;
    if (i0 >= n_self) return;
    const int head0 = d * B, tail0 = p.b_c0 + d * T, self0 = SIDE_B ? tail0 : head0, other0 = SIDE_B ? head0 : tail0;
    const char* const coef = p.in.coefp + (size_t)d * Bp * Tp * 6;
    const char* const a = SIDE_B ? coef + (size_t)(i0 >> 5) * 192 : coef + (size_t)i0 * Tp * 6;
    const char* const other = p.rows + (int64_t)other0 * pitch;
    const char* const b = other + (size_t)(kt0 >> 5) * 192;
    const uint32_t* const nflag = DIST == DIST_L2 ? p.nearflag + (size_t)d * MT * NT : nullptr;
    floatx16 acc[P::AM][P::AN];
#pragma unroll
    for (int m = 0; m < P::AM; ++m)
#pragma unroll
        for (int n = 0; n < P::AN; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
    uint32_t seen = 0u;  // flagged blocks among the tile's
    P::run(smem, a, Tp * 6, SIDE_B ? (size_t)32 * Tp * 6 : 192, b, pitch, (size_t)32 * pitch, n_slab, n_other, acc, lane, wave,
           [&]() __attribute__((always_inline)) {
               if (DIST != DIST_L2) return;
               // the self rows' coefficient sums, from the sub-blocks' in a fixed order
               for (int i = tid; i < TM; i += WM * WN * 64) {
                   float s = 0.f;
                   if (SIDE_B) {
                       if (i0 + i < Tp)
                           for (int q = 0; q < MT; ++q) s += p.in.colpart[((size_t)d * MT + q) * Tp + i0 + i];
                   } else if (i0 + i < Bp) {
                       for (int q = 0; q < n_slab; ++q) s += p.in.rowpart[((size_t)d * Bp + i0 + i) * NT + q];
                   }
                   csum_s[i] = s;
               }
               for (int x = tid; x < TM / 32 * n_slab; x += WM * WN * 64) {
                   const int st = (i0 >> 5) + x / n_slab, ot = x % n_slab;
                   if (SIDE_B ? st < NT : st < MT) seen |= SIDE_B ? nflag[(size_t)ot * NT + st] : nflag[(size_t)st * NT + ot];
               }
           });
    const int wm = (wave / WN) * (TM / WM), wn = (wave % WN) * (TN / WN);
    const int cl = lane & 31, hl = lane >> 5;
    const char* const self = p.rows + (int64_t)(self0 + i0) * pitch;
    if (DIST == DIST_L2 && __syncthreads_or(seen != 0u)) {
        // slabs in which some pair of a sub-block is nearly identical: c (self - other) directly, as
        // the reference codelet does (their coefficients went into the product as zeros; acc holds
        // the negated sum)
        const float* const cf = p.coef + (size_t)d * B * T;
#pragma unroll
        for (int mi = 0; mi < P::AM; ++mi)
            for (int ot = 0; ot < n_slab; ++ot) {
                const int st = (i0 + wm + 32 * mi) >> 5;
                if (st >= (SIDE_B ? NT : MT)) continue;
                if ((SIDE_B ? nflag[(size_t)ot * NT + st] : nflag[(size_t)st * NT + ot]) == 0u) continue;
#pragma unroll
                for (int ni = 0; ni < P::AN; ++ni) {
                    const int k = kt0 + wn + 32 * ni + cl;
                    if (kt0 + wn + 32 * ni >= p.Kp) continue;
                    float sv[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        sv[r] = load_piece1(self + (int64_t)(wm + 32 * mi + 8 * (r >> 2) + 4 * hl + (r & 3)) * pitch, k);
                    for (int j = 32 * ot; j < min(32 * ot + 32, n_other); ++j) {
                        const float o = load_piece1(other + (int64_t)j * pitch, k);
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int i = i0 + wm + 32 * mi + 8 * (r >> 2) + 4 * hl + (r & 3);
                            const float c = i < n_self ? (SIDE_B ? cf[(size_t)j * T + i] : cf[(size_t)i * T + j]) : 0.f;
                            acc[mi][ni][r] = fmaf(-c, sv[r] - o, acc[mi][ni][r]);
                        }
                    }
                }
            }
    }
    // neighbouring lanes swap values: a lane stores two columns of one row
    const bool odd = lane & 1;
    float* const out = p.grad + (size_t)(self0 + i0) * p.Dp;
#pragma unroll
    for (int mi = 0; mi < P::AM; ++mi)
#pragma unroll
        for (int ni = 0; ni < P::AN; ++ni) {
            const int k = kt0 + wn + 32 * ni + (cl & ~1);
            if (k >= p.Dp) continue;
            const char* const sp = self + (size_t)(k >> 5) * 192 + (k & 31) * 2;
            uint32_t w[DIST == DIST_L2 ? 8 : 1][3];
            if (DIST == DIST_L2)
#pragma unroll
                for (int i = 0; i < 8; ++i)  // all loads before any use, rows past the last among them
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        w[i][q] = *reinterpret_cast<const uint32_t*>(
                            sp + (int64_t)(wm + 32 * mi + 8 * (i >> 1) + 4 * hl + 2 * (i & 1) + odd) * pitch + 64 * q);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float got = swap1(odd ? acc[mi][ni][2 * i] : acc[mi][ni][2 * i + 1]);
                float x = odd ? got : acc[mi][ni][2 * i], y = odd ? acc[mi][ni][2 * i + 1] : got;
                const int row = wm + 32 * mi + 8 * (i >> 1) + 4 * hl + 2 * (i & 1) + odd;
                if (DIST == DIST_L2) {
                    float sx = 0.f, sy = 0.f;
#pragma unroll
                    for (int q = 0; q < 3; ++q) { sx += bf16_lo_f32(w[i][q]); sy += bf16_hi_f32(w[i][q]); }
                    x = sx * csum_s[row] - x;
                    y = sy * csum_s[row] - y;
                }
                if (i0 + row < n_self) *reinterpret_cast<float2*>(out + (size_t)row * p.Dp + k) = make_float2(x, y);
            }
        }
}

// Both sides in one launch: the side whose tiles loop over more rows comes first, for every block, so
// that the long tiles do not start last.  A block's tiles of one side stay together on one XCD.
template <int DIST>
__global__ __launch_bounds__(kWaves * kWaves * 64) void k_split_bwd(SplitBwd p) {
    constexpr int TM = kTile, TN = kTile;
    using PA = SplitProduct<RowTile<TM>, ColTile<TN>, TM, TN, kWaves, kWaves>;
    __shared__ __attribute__((aligned(16))) char smem[PA::kLds];
    __shared__ float csum_s[TM];
    const int gx = (p.Dp + TN - 1) / TN, ga = (p.B + TM - 1) / TM, gb = (p.T + TM - 1) / TM;
    const bool heads_first = p.T >= p.B;
    const int n_first = gx * (heads_first ? ga : gb) * p.S;
    const int L = blockIdx.x;
    if ((L < n_first) == heads_first) {
        const TileId tile = xcd_tile(gx, ga, p.S, heads_first ? L : L - n_first);
        split_bwd_tile<DIST, false>(p, tile.z, tile.x, tile.y, smem, csum_s);
    } else {
        const TileId tile = xcd_tile(gx, gb, p.S, heads_first ? L - n_first : L);
        split_bwd_tile<DIST, true>(p, tile.z, tile.x, tile.y, smem, csum_s);
    }
}

// --------------------------------------------------------------------------
// launches

int split_fwd_parts(const ScoreShape& sh) {
    return ((sh.T + kTile - 1) / kTile) * ((sh.B + kTile - 1) / kTile);
}

void launch_split_fwd(const SplitFwd& p, bool fused_loss, hipStream_t stream) {
    const ScoreShape& sh = p.sh;
    const dim3 grid = tile_grid((sh.T + kTile - 1) / kTile, (sh.B + kTile - 1) / kTile, sh.S);
    const bool l2 = sh.dist_fn == DIST_L2 && sh.score_fn != SCORE_DISTMULT;
#define KGE_FWD(D_, OM_) hipLaunchKernelGGL((k_split_fwd<D_, OM_>), grid, dim3(256), 0, stream, p)
    if (l2) { if (fused_loss) KGE_FWD(DIST_L2, 0); else KGE_FWD(DIST_L2, 1); }
    else    { if (fused_loss) KGE_FWD(DIST_DOT, 0); else KGE_FWD(DIST_DOT, 1); }
#undef KGE_FWD
}

void launch_coef_pieces(const ScoreShape& sh, const float* coef, const uint32_t* nearflag, const SplitCoef& out,
                        hipStream_t stream) {
    const int n = sh.S * (out.Bp / 32) * (out.Tp / 32);
    const bool l2 = sh.dist_fn == DIST_L2 && sh.score_fn != SCORE_DISTMULT;
    if (l2) hipLaunchKernelGGL(k_coef_pieces<DIST_L2>, dim3((n + 3) / 4), dim3(256), 0, stream, sh, coef, nearflag, out);
    else hipLaunchKernelGGL(k_coef_pieces<DIST_DOT>, dim3((n + 3) / 4), dim3(256), 0, stream, sh, coef, nearflag, out);
}

void launch_split_bwd(const SplitBwd& p, bool l2, hipStream_t stream) {
    const dim3 grid(((p.Dp + kTile - 1) / kTile) * ((p.B + kTile - 1) / kTile + (p.T + kTile - 1) / kTile) * p.S);
    if (l2) hipLaunchKernelGGL(k_split_bwd<DIST_L2>, grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL(k_split_bwd<DIST_DOT>, grid, dim3(256), 0, stream, p);
}

// Where these kernels are taken.  At whole 128-row tiles and enough of them the kernels that split
// float32 operands while staging are as fast or faster (22.8M-row workload, 64 blocks of 256 x 512:
// forward 40 against 42 us, backward 57 against 67, and the gather writes a third less): the
// piece matrices cost half as much memory traffic again, and with that many tiles the
// staging's vector work hides behind other workgroups' matrix work.  Elsewhere - ragged sizes, which
// those kernels take with bounds checks and float32 matrix instructions, and few tiles - these
// are the faster ones: one block of 256 x 64, D = 64: forward 11.2 -> 10.5 us, backward 37 -> 9.5;
// four of 200 x 268, D = 100: 17.4 -> 7.8 and 49 -> 10.6.
bool split_scoring(const ScoreShape& sh) {
    if (sh.use_mfma != 2 || sh.score_fn == SCORE_TRANSH) return false;
    if (sh.dist_fn == DIST_L1 && sh.score_fn != SCORE_DISTMULT) return false;
    const bool whole = sh.B % 128 == 0 && sh.T % 128 == 0 && sh.Dp % 64 == 0;
    return !whole || (int64_t)sh.S * (sh.B / 128) * (sh.T / 64) < 128;
}

}  // namespace kge
