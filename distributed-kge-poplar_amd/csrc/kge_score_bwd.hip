// gfx950 kernels of the scoring backward pass: l1 / l2distancegrad and the matMul backward
// (src/pag/pag.cpp:685-700, 777-836; the distance codelets of src/poplar_extensions).
#include "kge_device.h"

#include <algorithm>
#include <cstdint>

namespace kge {

// --------------------------------------------------------------------------
// scoring: backward.  out[i, k] = sum_j c[i, j] * phi(self[i, k], other[j, k])
//   L1   phi = signum(self - other)
//   L2   phi = self - other              (c already holds g / dist)
//   DOT  phi = other



template <int DIST>
__global__ __launch_bounds__(256) void k_score_bwd(BwdParams p) {
    __shared__ __attribute__((aligned(16))) float Cs[BJ][LDP];  // Cs[j][i]
    __shared__ __attribute__((aligned(16))) float Os[BJ][LDP];  // Os[j][k]
    const int B = p.B, T = p.T, Dp = p.Dp;
    const int n_self = p.side_b ? T : B;
    const TileId tile = xcd_tile((Dp + kScoreTile - 1) / kScoreTile, (n_self + kScoreTile - 1) / kScoreTile, p.S);
    const int d = tile.z, i0 = tile.y * kScoreTile, kt0 = tile.x * kScoreTile;
    const int t_live = tail_limit(p.tcount, d, T, p.tpad);  // merged tails: the block's live columns
    const int n_other = p.side_b ? B : t_live;
    if (p.side_b && i0 >= t_live) return;
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int self_c0 = (p.side_b ? p.b_c0 + d * T : p.a_c0 + d * B);
    const int other_c0 = (p.side_b ? p.a_c0 + d * B : p.b_c0 + d * T);
    const int self_rel = p.side_b ? 0 : p.a_rel_mode, other_rel = p.side_b ? p.a_rel_mode : 0;
    const RowSource& self_src = p.side_b ? p.ent_b : p.ent_a;
    const RowSource& other_src = p.side_b ? p.ent_a : p.ent_b;
    const float* coef = p.coef + (size_t)d * B * T;
    const float* cdiv = p.coef_div ? p.coef_div + (size_t)d * B * T : nullptr;

    // this thread's 4x4 block of `self` (needed by L1 in the loop, by L2 at the end)
    float sv[4][4];
    const int kcol = kt0 + tx * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = i0 + ty * 4 + i;
        float4 v = make_float4(0, 0, 0, 0);
        if (DIST != DIST_DOT && r < n_self && kcol < Dp) {
            v = load4(row_ptr(self_src, self_c0 + r), kcol, self_src);
            if (self_rel) v = combine_rel(v, p.rel + (size_t)p.crel[d * B + r] * Dp, kcol, self_rel);
        }
        sv[i][0] = v.x; sv[i][1] = v.y; sv[i][2] = v.z; sv[i][3] = v.w;
    }
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[i][k] = 0.f;

    for (int j0 = 0; j0 < n_other; j0 += BJ) {
        // coefficient tile -> Cs[j][i]
        if (!p.side_b) {
            // c[i][j] = coef[i0+i][j0+j], contiguous over j: transposing store
            const int li = tid >> 3, j4 = (tid & 7) * 4;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int i = li + 32 * h, gi = i0 + i, gj = j0 + j4;
                float v[4] = {0.f, 0.f, 0.f, 0.f};
                if (gi < B) {
                    const float* src = coef + (size_t)gi * T + gj;
                    if (cdiv) {
                        const float* dv = cdiv + (size_t)gi * T + gj;
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            if (gj + x < T) v[x] = dv[x] != 0.f ? src[x] / dv[x] : 0.f;
                    } else if (gj + 3 < T && (T & 3) == 0) {
                        const float4 t = *reinterpret_cast<const float4*>(src);
                        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
                    } else {
#pragma unroll
                        for (int x = 0; x < 4; ++x) if (gj + x < T) v[x] = src[x];
                    }
                }
#pragma unroll
                for (int x = 0; x < 4; ++x) Cs[j4 + x][i] = v[x];
            }
        } else {
            // c[i][j] = coef[j0+j][i0+i], contiguous over i: direct store
            const int lj = tid >> 4, i4 = (tid & 15) * 4;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int j = lj + 16 * h, gj = j0 + j, gi = i0 + i4;
                float4 t = make_float4(0, 0, 0, 0);
                if (gj < B) {
                    const float* src = coef + (size_t)gj * T + gi;
                    if (cdiv) {
                        const float* dv = cdiv + (size_t)gj * T + gi;
                        if (gi + 0 < T) t.x = dv[0] != 0.f ? src[0] / dv[0] : 0.f;
                        if (gi + 1 < T) t.y = dv[1] != 0.f ? src[1] / dv[1] : 0.f;
                        if (gi + 2 < T) t.z = dv[2] != 0.f ? src[2] / dv[2] : 0.f;
                        if (gi + 3 < T) t.w = dv[3] != 0.f ? src[3] / dv[3] : 0.f;
                    } else if (gi + 3 < T && (T & 3) == 0) {
                        t = *reinterpret_cast<const float4*>(src);
                    } else {
                        if (gi + 0 < T) t.x = src[0];
                        if (gi + 1 < T) t.y = src[1];
                        if (gi + 2 < T) t.z = src[2];
                        if (gi + 3 < T) t.w = src[3];
                    }
                }
                *reinterpret_cast<float4*>(&Cs[j][i4]) = t;
            }
        }
        // other rows -> Os[j][k]
        {
            const int lj = tid >> 4, kk4 = (tid & 15) * 4;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int j = lj + 16 * h, gj = j0 + j, gk = kt0 + kk4;
                float4 t = make_float4(0, 0, 0, 0);
                if (gj < n_other && gk < Dp) {
                    t = load4(row_ptr(other_src, other_c0 + gj), gk, other_src);
                    if (other_rel)
                        t = combine_rel(t, p.rel + (size_t)p.crel[d * B + gj] * Dp, gk, other_rel);
                }
                *reinterpret_cast<float4*>(&Os[j][kk4]) = t;
            }
        }
        __syncthreads();
#pragma unroll 8
        for (int jj = 0; jj < BJ; ++jj) {
            const float4 c4 = *reinterpret_cast<const float4*>(&Cs[jj][ty * 4]);
            const float4 o4 = *reinterpret_cast<const float4*>(&Os[jj][tx * 4]);
            const float cv[4] = {c4.x, c4.y, c4.z, c4.w};
            const float ov[4] = {o4.x, o4.y, o4.z, o4.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if (DIST == DIST_L1) {
                        const float t = sv[i][k] - ov[k];
                        const float sg = (t > 0.f ? 1.f : 0.f) - (t < 0.f ? 1.f : 0.f);
                        acc[i][k] = fmaf(cv[i], sg, acc[i][k]);
                    } else if (DIST == DIST_L2) {
                        acc[i][k] = fmaf(cv[i], sv[i][k] - ov[k], acc[i][k]);
                    } else {
                        acc[i][k] = fmaf(cv[i], ov[k], acc[i][k]);
                    }
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = i0 + ty * 4 + i;
        if (r >= n_self || kcol >= Dp) continue;
        float o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            o[k] = acc[i][k];
        }
        float* dst = p.grad + (size_t)(p.grad_c0 + d * n_self + r) * Dp + kcol;
        if (p.vec_out) {
            *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) if (kcol + k < Dp) dst[k] = o[k];
        }
    }
}

// --------------------------------------------------------------------------
// scoring backward on the matrix cores (L2 and dot):
//   out[i,k] = sum_j c[i,j] other[j,k]          (a [I x J] . [J x Dp] product)
//   L2: out[i,k] = self[i,k] * sum_j c[i,j] - that product
// Workgroup tile 128 (self rows) x 64 (embedding columns), waves 2 x 2, each
// wave two 32x32 accumulators; the next chunk of c and `other` is fetched into
// registers while the matrix cores work on the current one.

constexpr int BM_TI = 128, BM_TK = 64, BM_LDK = BM_TK + 4;
// LDS of a backward workgroup: two coefficient tiles (the larger layout: 128 x 36 floats),
// two `other` tiles (32 x 68 floats) and the 128 coefficient row sums
constexpr int kBwdSmemBytes = 2 * (BM_TI * 36 * 4) + 2 * (32 * BM_LDK * 4) + BM_TI * 4;

// BJT = rows of `other` staged per iteration (32 or 128) and NW = waves per
// workgroup (4 or 8), chosen as in the forward kernel.
// ALIGNED: n_self % 128 == 0, n_other % BJT == 0, Dp % 64 == 0, T % 4 == 0,
// dense float32 operands without a relation to apply: branch-free staging loads.
template <int DIST, int SIDE_B, int BJT, bool ALIGNED, int NW>
DEVINL void bwd_mfma_body(const BwdParams& p, const int d, const int tile_x, const int tile_y, char* smem) {
    // Both tiles are float4 copies of global memory.  Head side: Cs[i][j] (the
    // coefficient rows as stored), a lane reads four consecutive j of its row i
    // in one 16-byte LDS read.  Tail side: Cs[j][i] (coefficient rows are the
    // other operand's rows), a lane reads its column i of four rows j.
    constexpr int NT = NW * 64;
    constexpr int AT = 8 / NW;        // 32-row accumulator tiles per wave
    constexpr int NCH = BJT / 32;     // 32-row sub-chunks per iteration
    constexpr int HC = 1024 / NT;     // float4 of a 32 x 128 coefficient sub-tile per thread
    constexpr int HO = 512 / NT;      // float4 of a 32 x 64 `other` sub-tile per thread
    constexpr int CS_ROWS = SIDE_B ? BJT : BM_TI, CS_LD = SIDE_B ? BM_TI + 4 : BJT + 4;
    // two copies of each tile: while the matrix cores work on one slab the next is
    // staged into the other copy, with a single barrier per slab
    typedef float CsTile[CS_ROWS][CS_LD];
    typedef float OsTile[BJT][BM_LDK];
    static_assert(2 * sizeof(CsTile) + 2 * sizeof(OsTile) + BM_TI * 4 <= kBwdSmemBytes, "LDS carve-up");
    CsTile* Cs2 = reinterpret_cast<CsTile*>(smem);
    OsTile* Os2 = reinterpret_cast<OsTile*>(smem + 2 * sizeof(CsTile));
    float* csum_s = reinterpret_cast<float*>(smem + 2 * sizeof(CsTile) + 2 * sizeof(OsTile));
    const int i0 = tile_y * BM_TI, kt0 = tile_x * BM_TK;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave >> 1) * (32 * AT), wk = (wave & 1) * 32;
    const int B = p.B, T = p.T, Dp = p.Dp;
    const int t_live = tail_limit(p.tcount, d, T, p.tpad);  // merged tails: the block's live columns
    const int n_self = SIDE_B ? T : B, n_other = SIDE_B ? B : t_live;
    if (i0 >= (SIDE_B ? t_live : n_self)) return;  // the grid is sized for the longer side
    const int grad_c0 = SIDE_B ? p.b_c0 : p.a_c0;
    const int self_c0 = SIDE_B ? p.b_c0 + d * T : p.a_c0 + d * B;
    const int other_c0 = SIDE_B ? p.a_c0 + d * B : p.b_c0 + d * T;
    const int self_rel = SIDE_B ? 0 : p.a_rel_mode, other_rel = SIDE_B ? p.a_rel_mode : 0;
    const RowSource& self_src = SIDE_B ? p.ent_b : p.ent_a;
    const RowSource& other_src = SIDE_B ? p.ent_a : p.ent_b;
    const float* coef = p.coef + (size_t)d * B * T;

    floatx16 acc[AT];
#pragma unroll
    for (int t = 0; t < AT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
    float cs_acc = 0.f;
    constexpr int NQ = NT / BM_TI, QL = 32 / NQ;  // threads per coefficient row, coefficients per thread and slab
    const int crow = tid & (BM_TI - 1), cq = tid / BM_TI;
    const int kcol = kt0 + wk + (lane & 31);

    // L2: this lane's `self` values, in accumulator layout
    float sv[AT][16];
    if (DIST == DIST_L2) {
#pragma unroll
        for (int t = 0; t < AT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = i0 + wi + 32 * t + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (ALIGNED) {
                    sv[t][r] = reinterpret_cast<const float*>(
                        self_src.base + (int64_t)(self_c0 + i) * self_src.pitch)[kcol];
                    continue;
                }
                float v = 0.f;
                if (i < n_self && kcol < Dp) {
                    v = load1(row_ptr(self_src, self_c0 + i), kcol, self_src.etype);
                    if (self_rel) {
                        const float rv = p.rel[(size_t)p.crel[d * B + i] * Dp + kcol];
                        v = self_rel == 1 ? v + rv : v * rv;
                    }
                }
                sv[t][r] = v;
            }
    }
    // near-identical-pair flags of the (self sub-tile, other chunk) blocks
    const int MT = (B + 31) >> 5, NTL = (T + 31) >> 5;
    const uint32_t* nflag = (DIST == DIST_L2 && p.nearflag) ? p.nearflag + (size_t)d * MT * NTL : nullptr;
    auto flag_of = [&](int i_tile, int j_tile) -> uint32_t {
        if (!nflag) return 0u;
        const int mt = SIDE_B ? j_tile : i_tile, nt = SIDE_B ? i_tile : j_tile;
        if (32 * nt >= t_live) return 0u;  // columns the forward pass did not visit
        if (ALIGNED) return nflag[(size_t)mt * NTL + nt];
        return (mt < MT && nt < NTL) ? nflag[(size_t)mt * NTL + nt] : 0u;
    };
    uint32_t nf_next[NCH][AT], nf_row_next[NCH];
    floatx4 creg[NCH][HC], oreg[NCH][HO];
    auto prefetch = [&](int jbase) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int j0 = jbase + 32 * c;
#pragma unroll
            for (int t = 0; t < AT; ++t) nf_next[c][t] = flag_of((i0 + wi + 32 * t) >> 5, j0 >> 5);
            nf_row_next[c] = flag_of((i0 + (tid & (BM_TI - 1))) >> 5, j0 >> 5);
            if constexpr (ALIGNED) {
#pragma unroll
                for (int h = 0; h < HC; ++h) {
                    const int idx = tid + NT * h;
                    const float* src = SIDE_B ? coef + (size_t)(j0 + (idx >> 5)) * T + i0 + (idx & 31) * 4
                                              : coef + (size_t)(i0 + (idx >> 3)) * T + j0 + (idx & 7) * 4;
                    creg[c][h] = *reinterpret_cast<const floatx4*>(src);
                }
#pragma unroll
                for (int h = 0; h < HO; ++h) {
                    const int idx = tid + NT * h;
                    oreg[c][h] = *reinterpret_cast<const floatx4*>(
                        other_src.base + (int64_t)(other_c0 + j0 + (idx >> 4)) * other_src.pitch +
                        (size_t)(kt0 + (idx & 15) * 4) * 4);
                }
            } else {
#pragma unroll
            for (int h = 0; h < HC; ++h) {
                const int idx = tid + NT * h;
                creg[c][h] = floatx4{0.f, 0.f, 0.f, 0.f};
                if (!SIDE_B) {  // c[i][j] = coef[i0+i][j0+j]: float4 along j
                    const int gi = i0 + (idx >> 3), gj = j0 + (idx & 7) * 4;
                    if (gi < B && gj < T) {
                        const float* src = coef + (size_t)gi * T + gj;
                        if (gj + 3 < T && (T & 3) == 0) creg[c][h] = *reinterpret_cast<const floatx4*>(src);
                        else {
                            creg[c][h].x = src[0];
                            if (gj + 1 < T) creg[c][h].y = src[1];
                            if (gj + 2 < T) creg[c][h].z = src[2];
                            if (gj + 3 < T) creg[c][h].w = src[3];
                        }
                    }
                } else {        // c[i][j] = coef[j0+j][i0+i]: float4 along i
                    const int gj = j0 + (idx >> 5), gi = i0 + (idx & 31) * 4;
                    if (gj < B && gi < T) {
                        const float* src = coef + (size_t)gj * T + gi;
                        if (gi + 3 < T && (T & 3) == 0) creg[c][h] = *reinterpret_cast<const floatx4*>(src);
                        else {
                            creg[c][h].x = src[0];
                            if (gi + 1 < T) creg[c][h].y = src[1];
                            if (gi + 2 < T) creg[c][h].z = src[2];
                            if (gi + 3 < T) creg[c][h].w = src[3];
                        }
                    }
                }
            }
#pragma unroll
            for (int h = 0; h < HO; ++h) {
                const int idx = tid + NT * h;
                const int gj = j0 + (idx >> 4), gk = kt0 + (idx & 15) * 4;
                oreg[c][h] = floatx4{0.f, 0.f, 0.f, 0.f};
                if (gj < n_other && gk < Dp) {
                    oreg[c][h] = as_x4(load4(row_ptr(other_src, other_c0 + gj), gk, other_src));
                    if (other_rel)
                        oreg[c][h] = as_x4(combine_rel(as_f4(oreg[c][h]), p.rel + (size_t)p.crel[d * B + gj] * Dp, gk, other_rel));
                }
            }
            }
        }
    };
    bool direct_next[NCH][AT], direct_row_next[NCH], any_direct_next[NCH];
    // writes the prefetched slab into tile copy `nb` and latches its near-pair flags
    auto stage = [&](int nb) __attribute__((always_inline)) {
        CsTile& Cn = Cs2[nb];
        OsTile& On = Os2[nb];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            any_direct_next[c] = false;
#pragma unroll
            for (int t = 0; t < AT; ++t) {
                direct_next[c][t] = nf_next[c][t] != 0u;
                any_direct_next[c] = any_direct_next[c] || direct_next[c][t];
            }
            direct_row_next[c] = nf_row_next[c] != 0u;
#pragma unroll
            for (int h = 0; h < HC; ++h) {
                const int idx = tid + NT * h;
                if (!SIDE_B) {
                    *reinterpret_cast<floatx4*>(&Cn[idx >> 3][32 * c + (idx & 7) * 4]) = creg[c][h];
                } else {
                    *reinterpret_cast<floatx4*>(&Cn[32 * c + (idx >> 5)][(idx & 31) * 4]) = creg[c][h];
                }
            }
#pragma unroll
            for (int h = 0; h < HO; ++h) {
                const int idx = tid + NT * h;
                *reinterpret_cast<floatx4*>(&On[32 * c + (idx >> 4)][(idx & 15) * 4]) = oreg[c][h];
            }
        }
    };
    prefetch(0);
    stage(0);
    __syncthreads();
    if (BJT < n_other) prefetch(BJT);
    for (int jbase = 0, buf = 0; jbase < n_other; jbase += BJT, buf ^= 1) {
        bool direct[NCH][AT], direct_row[NCH], any_direct[NCH];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            any_direct[c] = any_direct_next[c];
            direct_row[c] = direct_row_next[c];
#pragma unroll
            for (int t = 0; t < AT; ++t) direct[c][t] = direct_next[c][t];
        }
        if (jbase + BJT < n_other) {
            stage(buf ^ 1);  // the other copy: last read one slab ago, before the barrier
            if (jbase + 2 * BJT < n_other) prefetch(jbase + 2 * BJT);
        }
        const CsTile& Cc = Cs2[buf];
        const OsTile& Oc = Os2[buf];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int jo = 32 * c;
            // coefficient row sums (L2): NQ threads share a row, each adds its QL of the slab's
            // 32 coefficients, so that every wave carries the same small load
            if (DIST == DIST_L2 && !direct_row[c]) {
                if (SIDE_B) {
#pragma unroll
                    for (int jj = 0; jj < QL; ++jj) cs_acc += Cc[jo + cq * QL + jj][crow];
                } else {
#pragma unroll
                    for (int jj = 0; jj < QL; jj += 4) {
                        const float4 v = *reinterpret_cast<const float4*>(&Cc[crow][jo + cq * QL + jj]);
                        cs_acc += v.x; cs_acc += v.y; cs_acc += v.z; cs_acc += v.w;
                    }
                }
            }
            if (!any_direct[c]) {
                // group g covers rows j = jo + 8g .. 8g+7 of `other`: instruction x
                // takes row 8g + x (lower half-wave) and 8g + 4 + x (upper)
                float ra[2][AT][4], rb[2][4];
                const int hl = lane >> 5, cl = lane & 31;
                auto fetch = [&](int buf, int g) {
#pragma unroll
                    for (int x = 0; x < 4; ++x) rb[buf][x] = Oc[jo + 8 * g + 4 * hl + x][wk + cl];
#pragma unroll
                    for (int t = 0; t < AT; ++t) {
                        if (SIDE_B) {
#pragma unroll
                            for (int x = 0; x < 4; ++x) ra[buf][t][x] = Cc[jo + 8 * g + 4 * hl + x][wi + 32 * t + cl];
                        } else {
                            const float4 v = *reinterpret_cast<const float4*>(&Cc[wi + 32 * t + cl][jo + 8 * g + 4 * hl]);
                            ra[buf][t][0] = v.x; ra[buf][t][1] = v.y; ra[buf][t][2] = v.z; ra[buf][t][3] = v.w;
                        }
                    }
                };
                fetch(0, 0);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    if (g + 1 < 4) fetch((g + 1) & 1, g + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int x = 0; x < 4; ++x)
#pragma unroll
                        for (int t = 0; t < AT; ++t)
                            acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[g & 1][t][x], rb[g & 1][x], acc[t], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                // some pair of this block is nearly identical: c * (self - other) directly,
                // as the reference codelet does (acc holds the negated sum, see the epilogue)
#pragma unroll
                for (int t = 0; t < AT; ++t) {
                    if (direct[c][t]) {
                        for (int jj = jo; jj < jo + 32; ++jj) {
                            const float o = Oc[jj][wk + (lane & 31)];
#pragma unroll
                            for (int r = 0; r < 16; ++r) {
                                const int il = wi + 32 * t + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                                const float cc = SIDE_B ? Cc[jj][il] : Cc[il][jj];
                                acc[t][r] = fmaf(-cc, sv[t][r] - o, acc[t][r]);
                            }
                        }
                    } else {
#pragma unroll
                        for (int q = 0; q < 16; ++q) {
                            const int jj = jo + 2 * q + (lane >> 5);
                            const float b = Oc[jj][wk + (lane & 31)];
                            const float a = SIDE_B ? Cc[jj][wi + 32 * t + (lane & 31)] : Cc[wi + 32 * t + (lane & 31)][jj];
                            acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[t], 0, 0, 0);
                        }
                    }
                }
            }
        }
        __syncthreads();
    }
    if (DIST == DIST_L2) {
        // the NQ partial sums of a row, added in a fixed order (the tiles are no longer read)
        float* part = reinterpret_cast<float*>(smem);
        part[cq * BM_TI + crow] = cs_acc;
        __syncthreads();
        if (tid < BM_TI) {
            float sum = part[tid];
#pragma unroll
            for (int q = 1; q < NQ; ++q) sum += part[q * BM_TI + tid];
            csum_s[tid] = sum;
        }
        __syncthreads();
    }
    float* __restrict__ const gout = p.grad;
    if (DIST == DIST_DOT && p.add_base) {
        // added rows: all row ids, then all values, then the stores, so that a tile's loads are
        // in flight together instead of sixteen dependent round trips one after the other
        const char* __restrict__ const ab = p.add_base;
        const uint32_t* __restrict__ const ai = p.add_index;
        const uint32_t cnt = *p.add_count;
#pragma unroll
        for (int t = 0; t < AT; ++t) {
            uint32_t row[16];
            float addv[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = i0 + wi + 32 * t + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                row[r] = ((ALIGNED || i < n_self) && (uint32_t)i < cnt) ? ai[i] : 0u;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r)
                addv[r] = (ALIGNED || kcol < Dp) ? load1(ab + (int64_t)row[r] * p.add_pitch, kcol, p.add_etype) : 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = i0 + wi + 32 * t + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (!ALIGNED && (i >= n_self || kcol >= Dp)) continue;
                gout[(size_t)(grad_c0 + d * n_self + i) * Dp + kcol] = acc[t][r] + addv[r];
            }
        }
        return;
    }
#pragma unroll
    for (int t = 0; t < AT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i_loc = wi + 32 * t + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            const int i = i0 + i_loc;
            if (!ALIGNED && (i >= n_self || kcol >= Dp)) continue;
            float o = acc[t][r];
            if (DIST == DIST_L2) o = sv[t][r] * csum_s[i_loc] - o;
            gout[(size_t)(grad_c0 + d * n_self + i) * Dp + kcol] = o;
        }
}

// one side per launch (p.side_b), or both sides in one launch
template <int DIST, int SIDE_B, int BJT, bool ALIGNED, int NW>
__global__ __launch_bounds__(NW * 64) void k_score_bwd_mfma(BwdParams p) {
    __shared__ __attribute__((aligned(16))) char smem[kBwdSmemBytes];
    const int n_self = SIDE_B ? p.T : p.B;
    const TileId tile = xcd_tile((p.Dp + BM_TK - 1) / BM_TK, (n_self + BM_TI - 1) / BM_TI, p.S);
    bwd_mfma_body<DIST, SIDE_B, BJT, ALIGNED, NW>(p, tile.z, tile.x, tile.y, smem);
}
template <int DIST, int BJT, bool ALIGNED, int NW>
__global__ __launch_bounds__(NW * 64) void k_score_bwd_mfma_both(BwdParams p) {
    __shared__ __attribute__((aligned(16))) char smem[kBwdSmemBytes];  // one allocation serves either side
    // One launch for both sides. The side whose tiles loop over more rows of the other side comes
    // first, for every block, then the other side: the long tiles do not start last (at the end of
    // the launch the CUs run dry while the longest tiles finish), and no workgroup is started for
    // a tile that does not exist. A block's tiles of one side stay together on one XCD; its two
    // sides no longer run close enough in time to share the L2's copy of the operand rows and the
    // coefficient matrix, which was measured to cost less than the late long tiles did.
    const int gx = p.Dp / BM_TK, ga = p.B / BM_TI, gb = p.T / BM_TI;
    const bool heads_first = p.T >= p.B;  // a head tile loops over T rows, a tail tile over B
    const int n_first = gx * (heads_first ? ga : gb) * p.S;
    const int L = blockIdx.x;
    if ((L < n_first) == heads_first) {
        const TileId tile = xcd_tile(gx, ga, p.S, heads_first ? L : L - n_first);
        bwd_mfma_body<DIST, 0, BJT, ALIGNED, NW>(p, tile.z, tile.x, tile.y, smem);
    } else {
        const TileId tile = xcd_tile(gx, gb, p.S, heads_first ? L - n_first : L);
        bwd_mfma_body<DIST, 1, BJT, ALIGNED, NW>(p, tile.z, tile.x, tile.y, smem);
    }
}

// --------------------------------------------------------------------------
// The same sums of a dot product (TransH's, and DistMult's where bfloat16 scoring meets shapes that its own products do
// not take) from bfloat16 matrix instructions on three-piece operands (mfma_split6: six
// v_mfma_f32_32x32x16_bf16 per sixteen rows of `other` in place of eight
// v_mfma_f32_32x32x2_f32, float32 accuracy).  The sum runs over the rows of `other`, so both
// operand tiles are laid down in LDS with that index innermost, as pieces:
//   Ap[piece][self row][32 j]    Bp[piece][embedding column][32 j]
// A thread stages eight consecutive j of one coefficient row (head side: two 16-byte loads along
// the row; tail side: eight 4-byte loads down a column of the coefficient matrix, consecutive
// lanes on consecutive columns) and four consecutive j of one embedding column of `other`.
// A row's four 16-byte chunks sit at position chunk ^ ((row / 4) % 4), which spreads sixteen
// consecutive rows' accesses to one chunk over all banks.
// Workgroup tile 128 (self rows) x 64 (embedding columns), eight waves as 4 x 2, one 32 x 32
// accumulator each; tile-aligned shapes and dense float32 operands only.

constexpr int BS_TI = 128, BS_TK = 64, BS_KJ = 32;
constexpr int kBwdSplitSmemBytes = 2 * 3 * BS_TI * BS_KJ * 2 + 2 * 3 * BS_TK * BS_KJ * 2;

template <int SIDE_B>
DEVINL void bwd_split_body(const BwdParams& p, const int d, const int tile_x, const int tile_y, char* smem) {
    typedef uint16_t ATile[3][BS_TI][BS_KJ];
    typedef uint16_t BTile[3][BS_TK][BS_KJ];
    ATile* Ap = reinterpret_cast<ATile*>(smem);
    BTile* Bp = reinterpret_cast<BTile*>(smem + 2 * sizeof(ATile));
    const int i0 = tile_y * BS_TI, kt0 = tile_x * BS_TK;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hl = lane >> 5, cl = lane & 31;
    const int wi = (wave >> 1) * 32, wk = (wave & 1) * 32;
    const int B = p.B, T = p.T, Dp = p.Dp;
    const int t_live = tail_limit(p.tcount, d, T, p.tpad);  // merged tails: the block's live columns
    const int n_self = SIDE_B ? T : B, n_other = SIDE_B ? B : t_live;
    if (i0 >= (SIDE_B ? t_live : n_self)) return;  // the grid is sized for the longer side
    const int grad_c0 = SIDE_B ? p.b_c0 : p.a_c0;
    const RowSource& other_src = SIDE_B ? p.ent_a : p.ent_b;
    const char* const other_rows = other_src.base + (int64_t)(SIDE_B ? p.a_c0 + d * B : p.b_c0 + d * T) * other_src.pitch;
    const int64_t opitch = other_src.pitch;
    const float* const coef = p.coef + (size_t)d * B * T;
    const int kcol = kt0 + wk + cl;

    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    // staging: coefficient row a_row, its j-chunk a_kg (8 values); column b_n of `other`, rows
    // 8 b_kg + 4 b_half .. + 3 of the slab.  What is the same for a whole wave stays in scalar
    // registers, so that the loads take a scalar base and one 32-bit lane offset.
    const int a_row = SIDE_B ? (wave & 1) * 64 + lane : wave * 16 + (lane >> 2), a_kg = SIDE_B ? (wave >> 1) : (lane & 3);
    const int b_n = lane, b_kg = wave & 3, b_half = wave >> 2;
    const int a_col = (a_kg ^ ((a_row >> 2) & 3)) << 3;
    const int b_col = ((b_kg ^ ((b_n >> 2) & 3)) << 3) + 4 * b_half;
    const uint32_t a_off = SIDE_B ? (uint32_t)a_row : (uint32_t)(a_row * T + 8 * a_kg);
    // a slab's operand loads take a round trip to the memory-side cache however little work a
    // slab is: two register sets, each filled two slabs ahead of its use
    struct Slab { floatx4 a[2], b; } set0, set1;
    auto prefetch = [&](Slab& s, int j_first) __attribute__((always_inline)) {
        // (taken through a scalar register afresh: the row addresses are then formed by scalar
        // instructions every slab, not carried along as one 64-bit vector pointer per row)
        const int j0 = __builtin_amdgcn_readfirstlane(j_first);
        if (!SIDE_B) {
            const float* src = coef + (size_t)i0 * T + j0;
            s.a[0] = *reinterpret_cast<const floatx4*>(src + a_off);
            s.a[1] = *reinterpret_cast<const floatx4*>(src + a_off + 4);
        } else {
#pragma unroll
            for (int x = 0; x < 8; ++x) s.a[x >> 2][x & 3] = (coef + (size_t)(j0 + 8 * a_kg + x) * T + i0)[a_off];
        }
#pragma unroll
        for (int x = 0; x < 4; ++x)
            s.b[x] = (reinterpret_cast<const float*>(other_rows + (int64_t)(j0 + 8 * b_kg + 4 * b_half + x) * opitch) + kt0)[b_n];
    };
    // writes a prefetched slab into tile copy `nb` as pieces; `live` = 0 for a slab past the end
    auto stage = [&](const Slab& s, int nb, float live) __attribute__((always_inline)) {
        const floatx4 a0 = s.a[0] * live, a1 = s.a[1] * live;
        uint2 lo[3], hi[3];
        split4_bf16(a0, lo);
        split4_bf16(a1, hi);
#pragma unroll
        for (int q = 0; q < 3; ++q)
            *reinterpret_cast<uint4*>(&Ap[nb][q][a_row][a_col]) = make_uint4(lo[q].x, lo[q].y, hi[q].x, hi[q].y);
        uint2 pb[3];
        split4_bf16(s.b, pb);
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(&Bp[nb][q][b_n][b_col]) = pb[q];
    };
    const int j_last = n_other - BS_KJ;  // loads past the end fetch the last slab again
    // one slab: the matrix work on tile copy `buf`, the next slab (register set `s`) into the
    // other copy (last read one slab ago, before the barrier), and `s` filled again
    auto step = [&](Slab& s, int jbase, int buf) __attribute__((always_inline)) {
        // two steps of sixteen rows of `other`; a lane supplies rows 8 * (lane / 32) .. + 7 of a
        // step, for its self row and for its embedding column
        floatx4 fa[2][3], fb[2][3];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int chunk = 2 * ks + hl;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int ra = wi + cl, rb = wk + cl;
                fa[ks][q] = *reinterpret_cast<const floatx4*>(&Ap[buf][q][ra][(chunk ^ ((ra >> 2) & 3)) << 3]);
                fb[ks][q] = *reinterpret_cast<const floatx4*>(&Bp[buf][q][rb][(chunk ^ ((rb >> 2) & 3)) << 3]);
            }
        }
        stage(s, buf ^ 1, jbase + BS_KJ < n_other ? 1.f : 0.f);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) acc = mfma_split6(fa[ks], fb[ks], acc);
        // the order asked of the scheduler: the first step's LDS reads, then one matrix
        // instruction (each depends on the one before it), a share of the vector work and an LDS
        // access, in turn
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
        for (int i = 0; i < 12; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);
            if (i < 6) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            else __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
        prefetch(s, min(jbase + 3 * BS_KJ, j_last));
        __syncthreads();
    };
    prefetch(set0, 0);
    stage(set0, 0, 1.f);
    prefetch(set0, min(BS_KJ, j_last));
    prefetch(set1, min(2 * BS_KJ, j_last));
    __syncthreads();
    for (int jbase = 0; jbase < n_other; jbase += 2 * BS_KJ) {  // n_other % 64 == 0
        step(set0, jbase, 0);
        step(set1, jbase + BS_KJ, 1);
    }
    float* __restrict__ const gout = p.grad;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int i_loc = wi + 8 * (r >> 2) + 4 * hl + (r & 3);
        gout[(size_t)(grad_c0 + d * n_self + i0 + i_loc) * Dp + kcol] = acc[r];
    }
}

// both sides in one launch, in the order of k_score_bwd_mfma_both
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_score_bwd_split_both(BwdParams p) {
    __shared__ __attribute__((aligned(16))) char smem[kBwdSplitSmemBytes];
    const int gx = p.Dp / BS_TK, ga = p.B / BS_TI, gb = p.T / BS_TI;
    const bool heads_first = p.T >= p.B;  // a head tile loops over T rows, a tail tile over B
    const int n_first = gx * (heads_first ? ga : gb) * p.S;
    const int L = blockIdx.x;
    if ((L < n_first) == heads_first) {
        const TileId tile = xcd_tile(gx, ga, p.S, heads_first ? L : L - n_first);
        bwd_split_body<0>(p, tile.z, tile.x, tile.y, smem);
    } else {
        const TileId tile = xcd_tile(gx, gb, p.S, heads_first ? L - n_first : L);
        bwd_split_body<1>(p, tile.z, tile.x, tile.y, smem);
    }
}

void launch_bwd(const BwdParams& p, int dist_fn, hipStream_t stream) {
    const int n_self = p.side_b ? p.T : p.B;
    const bool mfma_ok = p.use_mfma && !p.coef_div && p.ent_a.vec && p.ent_b.vec && (p.Dp & 3) == 0 &&
                         (dist_fn == DIST_DOT || (dist_fn == DIST_L2 && p.nearflag));
    if (mfma_ok) {
        const dim3 grid = tile_grid((p.Dp + BM_TK - 1) / BM_TK, (n_self + BM_TI - 1) / BM_TI, p.S);
        const int n_other = p.side_b ? p.B : p.T;
        const bool plain = p.ent_a.etype == ET_F32 && p.ent_b.etype == ET_F32 && !p.ent_a.index &&
                           !p.ent_b.index && p.a_rel_mode == 0;
        const bool aligned = plain && n_self % BM_TI == 0 && p.Dp % BM_TK == 0 && p.T % 4 == 0 && n_other % 32 == 0;
#define KGE_BWD(D_, S_)                                                                                     \
    do {                                                                                                    \
        if (aligned) hipLaunchKernelGGL((k_score_bwd_mfma<D_, S_, 32, true, 8>), grid, dim3(512), 0, stream, p); \
        else hipLaunchKernelGGL((k_score_bwd_mfma<D_, S_, 32, false, 4>), grid, dim3(256), 0, stream, p);    \
    } while (0)
        if (dist_fn == DIST_L2) {
            if (p.side_b) KGE_BWD(DIST_L2, 1); else KGE_BWD(DIST_L2, 0);
        } else {
            if (p.side_b) KGE_BWD(DIST_DOT, 1); else KGE_BWD(DIST_DOT, 0);
        }
#undef KGE_BWD
        return;
    }
    const dim3 grid = tile_grid((p.Dp + kScoreTile - 1) / kScoreTile, (n_self + kScoreTile - 1) / kScoreTile, p.S);
    if (dist_fn == DIST_L1)
        hipLaunchKernelGGL(k_score_bwd<DIST_L1>, grid, dim3(256), 0, stream, p);
    else if (dist_fn == DIST_L2)
        hipLaunchKernelGGL(k_score_bwd<DIST_L2>, grid, dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL(k_score_bwd<DIST_DOT>, grid, dim3(256), 0, stream, p);
}


// --------------------------------------------------------------------------
// L1 backward, both sides in one pass over the pairs, at any shape.  c * signum(a - b) has no
// contraction form, so this is vector-ALU work; computing the term once and
// adding it to the head's sum and (negated) to the tail's sum halves it.
// One workgroup of 16 waves per (block, 64-column slice, group of heads, group of at most 512
// tails: l1_pair_split); a lane owns one column.  Wave w keeps tails [w*tw, (w+1)*tw) of the
// group and their gradient sums in registers and walks over the group's heads; a head's sum over one wave's tails is a
// partial, the 16 partials of a head meet in LDS and are added in a fixed order.
// The coefficients of a (head, tail) are the same for every lane: a wave brings those of eight heads and
// its own tails to LDS (one to four per lane; the next chunk's in flight under the current one's
// arithmetic) and reads them four at a time with one instruction whose lanes all name the same address (a broadcast:
// 4 cycles per CU).  As scalar operands the same coefficients halve the rate of the instructions that take them.
constexpr int L1P_CB = 8;      // heads per chunk
constexpr int L1P_WAVES = 16;

constexpr int L1P_MAX_T = 512;  // tails per workgroup at most (32 per wave)

// One workgroup's share of a block: its heads, its tails, its 64 columns.
struct L1Pair {
    const float* a_rows;  // the first head's value in the block's first column; rows Dp apart
    const float* b_rows;  // the first tail's
    const float* coef;    // coefficient of the first head and the first tail; rows `ldc` apart
    float* grad_a;        // where the first head's gradient in the block's first column goes
    float* grad_b;
    int n_head, n_tail, ldc, Dp;
    int k0, kc;           // the slice's first column, this lane's column
    bool col;             // this lane has a column (another lane's otherwise)
};

// What the workgroup keeps in LDS: every wave's coefficients of a chunk and half their column sums
// (nobody else's business), and the heads' partial sums.
struct L1PairLds {
    float cs[L1P_WAVES][2][L1P_CB][L1P_MAX_T / L1P_WAVES];
    float col_half[L1P_WAVES][L1P_MAX_T / L1P_WAVES];
    float part[2][L1P_WAVES][L1P_CB][64];
};

template <int CTRL>
DEVINL float dpp_f32(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// the work of one wave with exactly TW tails (TW even): straight-line code over
// its tails, their values and sums in registers.
// signum(a - b) with signum(0) = 0 (poplar_extensions l1distance.codelet.cpp:76-79) from
// instructions of the fast class only (subtract, fused multiply-add): the difference times 2^126
// plus one half, clamped to [0, 1] by the instruction's own output modifier, is p = 1 / 0.5 / 0
// for a positive / zero / negative difference (any normal float times 2^126 is at least 1 in
// magnitude), and signum = 2 p - 1.  The inner loop accumulates c p (four instructions per pair
// and column: subtract, clamped fma, one fma for either side's sum) and the linear part is taken
// off in small pieces, before the sums grow and rounding with them:
//   tails   after every chunk of 8 heads, half the chunk's column sums: the running value is
//           sum c (p - 1/2) = (1/2) sum c signum;
//   heads   each wave's partial 2 sum_j c p minus the sum of the coefficients of its own TW
//           columns, before the 16 waves' values are added.
// Either linear part is summed in the order of the multiply-adds that it is taken from, so that a column in
// which heads and tails are equal (p = 1/2 throughout: the padding, rows of zeros) comes out as exactly zero.
// Bound by vector issue.  A head's sum runs in four chains: in one chain every multiply-add waits for
// the one before, and four waves per SIMD do not fill that gap (a register-only loop of these
// four instructions: 3.05 cycles of 2.4 GHz per instruction with one chain, 2.25 with four).  Everything
// but the heads' partial sums belongs to a wave alone, is asked for a chunk ahead, and is worked off between the
// heads; one barrier per chunk.  64 blocks of 256 x 512 (331 distinct tails each), D = 256: 147 -> 132 us; 16 of 512 x 1536:
// 315 -> 284.  2.6 cycles per instruction, of which one in seven is not the pairs' own; the rest of the launch
// is waiting for the block with the most distinct tails (7 % above their mean) and for its start and end.
// FULL: whole chunks of heads, 8-byte coefficient loads, readable zero coefficients up to the next
// multiple of 32 tails and a column in every lane: no bounds checks.
template <int TW, bool FULL>
DEVINL void l1_pair_wave(const L1Pair& q, int w, int lane, L1PairLds& lds) {
    constexpr int TWM = L1P_MAX_T / L1P_WAVES;
    // The widest copies have no register for what can be had again: heads' values are asked for eight (a chunk), four or
    // two heads ahead, and places that follow from the lane are formed where they are used.  (Copies
    // that have the registers are up to 7 % slower so.)  Nothing goes to scratch: 64 blocks of 250 x 512 distinct tails,
    // D = 256: 243 -> 221 us, 32 of 250 x 480: 118 -> 110; of whole groups the same as with scratch.
    constexpr int AHEAD = TW < 28 ? L1P_CB : TW < 32 ? 4 : 2;
    auto lane_again = [&]() __attribute__((always_inline)) { return TW < 30 ? (uint32_t)lane : lane_here(); };
    const int n_head = q.n_head, t0 = w * TW;
    const size_t Dp = q.Dp;
    // staging: lane -> (head, CPL columns) of the wave's coefficients of a chunk.  Loads without a branch
    // (a lane that has nothing to fetch fetches something else: a load that may not have been issued would be
    // waited for together with what was asked for before it); what does not count becomes zero when it has come.
    // A narrow copy's eight lanes per head take as many columns as the wave has tails for: with four each, most lanes of
    // most loads brought nothing, and the loads' addresses bounded the short loops (one block of 40 x 1500,
    // D = 256, up to 8 tails per wave: 13.5 -> 11.7 us; 4 of 200 x 268, D = 100: 14.5 -> 13.0; 33 x 90, D = 30: 11.7 -> 10.3).
    constexpr int CPL = TW <= 8 ? 1 : TW <= 16 ? 2 : 4;
    const int s_head = lane >> 3, s_col = (lane & 7) * CPL;
    const int s_n = (FULL ? TW : min(TW, q.n_tail - t0)) - s_col;  // columns of this lane that count
    struct Coefs { float v[CPL]; };
    auto fetch = [&](int b0) __attribute__((always_inline)) {
        const uint32_t l = lane_again(), head = l >> 3, col = (l & 7) * CPL;
        Coefs c;
        // the chunk's first row and the wave's first column in scalar registers, what is the lane's in 32 bits
        if constexpr (FULL) {
            const float* src = q.coef + (size_t)b0 * q.ldc + t0;
            const uint32_t row = head * (uint32_t)q.ldc;
            constexpr int N = CPL > 1 ? 2 : 1;
#pragma unroll
            for (int i = 0; i < CPL; i += N) {
                const float* at = src + (row + (col + i < TW ? col + i : 0u));
                if constexpr (N == 1) c.v[0] = at[0];
                else {
                    const float2 two = *reinterpret_cast<const float2*>(at);
                    c.v[i] = two.x; c.v[i + 1] = two.y;
                }
            }
        } else {
            const int b = min(b0, n_head - 1), t = min(t0, q.n_tail - 1);
            const float* src = q.coef + (size_t)b * q.ldc + t;
            const uint32_t row = min(head, (uint32_t)(n_head - 1 - b)) * (uint32_t)q.ldc, last = q.n_tail - 1 - t;
#pragma unroll
            for (int i = 0; i < CPL; ++i) c.v[i] = src[row + min(col + i, last)];
        }
        return c;
    };
    // a chunk's coefficients into the wave's tile `buf`
    auto stage = [&](int buf, int b0, Coefs c) __attribute__((always_inline)) {
        const int n = FULL || b0 + s_head < n_head ? s_n : 0;
        float* const to = &lds.cs[w][buf][s_head][s_col];
#pragma unroll
        for (int i = 0; i < CPL; ++i) if (n <= i) c.v[i] = 0.f;
        if constexpr (CPL == 4) *reinterpret_cast<float4*>(to) = make_float4(c.v[0], c.v[1], c.v[2], c.v[3]);
        else if constexpr (CPL == 2) *reinterpret_cast<float2*>(to) = make_float2(c.v[0], c.v[1]);
        else *to = c.v[0];
    };
    // the sums of a chunk's coefficients per head (the same in the head's eight lanes)
    constexpr int NG = (TW + 3) / 4;
    auto row_sums = [&](int buf) __attribute__((always_inline)) {
        const float* c = &lds.cs[w][buf][s_head][lane & 3];
        float r = c[0];
#pragma unroll
        for (int g = 1; g < NG; ++g) r += c[4 * g];
        r += dpp_f32<0xB1>(r);  // lane ^ 1
        r += dpp_f32<0x4E>(r);  // lane ^ 2
        return r;
    };
    // (the row's address in scalar registers: one 32-bit lane offset serves all loads)
    auto head_value = [&](int b) __attribute__((always_inline)) {
        typedef const __attribute__((address_space(1))) float* global_row;
        global_row row = (global_row)q.a_rows + (size_t)__builtin_amdgcn_readfirstlane(FULL ? b : min(b, n_head - 1)) * Dp;
        asm("" : "+s"(row));
        return row[(uint32_t)q.kc];
    };
    float bt[TW], gt[TW];
#pragma unroll
    for (int j = 0; j < TW; ++j) {
        bt[j] = (q.b_rows + (size_t)(FULL ? t0 + j : min(t0 + j, q.n_tail - 1)) * Dp)[(uint32_t)q.kc];
        gt[j] = 0.f;
    }
    // sixteen partials of a head: wave w takes head w / 2 of the chunk and half of the columns, the lower lanes the
    // first eight waves' partials, the upper ones the others'
    const int r_head = w >> 1;
    float red[8];
    auto ask = [&](int buf) __attribute__((always_inline)) {
        const uint32_t l = lane_again(), r_wave = (l >> 5) * 8, r_col = (w & 1) * 32 + (l & 31);
#pragma unroll
        for (int v = 0; v < 8; ++v) red[v] = lds.part[buf][r_wave + v][r_head][r_col];
    };
    auto give = [&](int b0) __attribute__((always_inline)) {
        float sum = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
        sum += __shfl_xor(sum, 32, 64);
        const uint32_t l = lane_again(), r_col = (w & 1) * 32 + (l & 31);
        const int b = b0 + r_head;
        if (l < 32 && (FULL || q.k0 + (int)r_col < q.Dp) && b >= 0 && (FULL || b < n_head))
            (q.grad_a + (size_t)b * Dp + q.k0)[r_col] = sum;
    };
    stage(0, 0, fetch(0));
    wave_lds_fence();
    float row_sum = row_sums(0);
    lds.col_half[w][lane & (TWM - 1)] = 0.f;
    float a[AHEAD];
#pragma unroll
    for (int h = 0; h < AHEAD; ++h) a[h] = head_value(h);
    // (waited for here: the loop's waits then count on the loop's own order of loads)
#pragma unroll
    for (int h = 0; h < AHEAD; ++h) asm volatile("" : "+v"(a[h]));
#pragma unroll
    for (int j = 0; j < TW; ++j) asm volatile("" : "+v"(bt[j]));
    int buf = 0, b0 = 0;
    for (; b0 < n_head; b0 += L1P_CB, buf ^= 1) {
        const int next = FULL ? min(b0 + L1P_CB, n_head - L1P_CB) : b0 + L1P_CB;  // (past the end: never used)
        Coefs c_next = fetch(next);
        float next_sum = 0.f;
        wave_lds_fence();
        // four tails at a time, their coefficients read two groups ahead; the order of the groups is kept
        // (left to itself the scheduler runs the heads into one another and out of registers)
        float4 c4[3];
        c4[0] = *reinterpret_cast<const float4*>(&lds.cs[w][buf][0][0]);
        c4[1] = *reinterpret_cast<const float4*>(&lds.cs[w][buf][1 / NG][(1 % NG) * 4]);
        float col[L1P_CB];
        float4 half = *reinterpret_cast<const float4*>(&lds.col_half[w][0]);
#pragma unroll
        for (int h = 0; h < L1P_CB; ++h) {
            // A wave that is behind goes first: left to themselves a SIMD's waves finish the chunk one after the
            // other, and the last one, alone, issues at half the rate (4.3 cycles per instruction against
            // 2.3 with company).
            if (h == 0) __builtin_amdgcn_s_setprio(3);
            if (h == 3) __builtin_amdgcn_s_setprio(2);
            if (h == 6) __builtin_amdgcn_s_setprio(1);
            if (h == 7) __builtin_amdgcn_s_setprio(0);
            // what is not the pairs' own work, each part's operands asked for a head before they are used, so that
            // nothing but the barrier stands between two chunks: the heads' sums of the chunk before, this
            // chunk's column sums, the next chunk's coefficients
            if (h == 1) ask(buf ^ 1);
            if (h == 2) give(b0 - L1P_CB);
            if (h == 3)
#pragma unroll
                for (int i = 0; i < L1P_CB; ++i) col[i] = lds.cs[w][buf][i][lane & (TWM - 1)];
            if (h == 4) {  // (both halves of the wave: the same value)
                lds.col_half[w][lane & (TWM - 1)] =
                    0.5f * (((((((col[0] + col[1]) + col[2]) + col[3]) + col[4]) + col[5]) + col[6]) + col[7]);
            }
            if (h == 6) {
#pragma unroll
                for (int i = 0; i < CPL; ++i) asm volatile("" : "+v"(c_next.v[i]));  // (not before)
                stage(buf ^ 1, next, c_next);
                wave_lds_fence();
            }
            if (h == 7) next_sum = row_sums(buf ^ 1);
            float gp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j4 = 0; j4 < TW; j4 += 4) {
                const int g = h * NG + j4 / 4, ahead = min(g + 2, L1P_CB * NG - 1);
                c4[(g + 2) % 3] = *reinterpret_cast<const float4*>(&lds.cs[w][buf][ahead / NG][(ahead % NG) * 4]);
                const float cv[4] = {c4[g % 3].x, c4[g % 3].y, c4[g % 3].z, c4[g % 3].w};
                float d[4], p[4];
                if (h == 0) {  // the chunk before's
                    const float hv[4] = {half.x, half.y, half.z, half.w};
#pragma unroll
                    for (int x = 0; x < 4; ++x) if (j4 + x < TW) gt[j4 + x] -= hv[x];
                    half = *reinterpret_cast<const float4*>(&lds.col_half[w][min(j4 + 4, TWM - 4)]);
                }
#pragma unroll
                for (int x = 0; x < 4; ++x) d[x] = a[h % AHEAD] - bt[min(j4 + x, TW - 1)];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int x = 0; x < 4; ++x) p[x] = __builtin_amdgcn_fmed3f(fmaf(d[x], 0x1p126f, 0.5f), 0.f, 1.f);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    if (j4 + x >= TW) continue;
                    gp[x] = fmaf(cv[x], p[x], gp[x]);
                    gt[j4 + x] = fmaf(cv[x], p[x], gt[j4 + x]);
                    asm volatile("" : "+v"(gt[j4 + x]));  // (not put off to the end of the chunk)
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            a[h % AHEAD] = head_value(h + AHEAD < L1P_CB ? b0 + h + AHEAD : next + h + AHEAD - L1P_CB);
            const float rs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(row_sum), h * 8));
            lds.part[buf][w][h][lane] = fmaf(2.f, (gp[0] + gp[1]) + (gp[2] + gp[3]), -rs);
        }
        row_sum = next_sum;
        __syncthreads();
    }
    ask(buf ^ 1);
    give(b0 - L1P_CB);
    const uint32_t kl = lane_again();
#pragma unroll
    for (int j = 0; j < TW; ++j)
        if (FULL || (t0 + j < q.n_tail && q.k0 + (int)kl < q.Dp))
            (q.grad_b + (size_t)(t0 + j) * Dp + q.k0)[kl] = -2.f * (gt[j] - lds.col_half[w][j]);
}

// How a block's pairs are divided: `heads` x `tails` groups, every group a workgroup per 64 columns.
// A group holds at most 512 tails.  A split leaves the other side's sums in pieces, which
// k_l1_pair_sum adds up: heads' gradients in `tails` pieces [tails][S * B][Dp], then the tails' in
// `heads` pieces [heads][S * T][Dp].
struct L1Split { int heads, tails; };
static L1Split l1_pair_split(const ScoreShape& sh) {
    // A workgroup of sixteen waves fills a CU.  Of the group sizes that the kernel has loops for, with
    // as many groups of heads (four chunks of eight at least) as the chip then has CUs left, the one whose
    // workgroups are done first: heads of a group times tails per wave and kHead, what a head costs
    // beside its tails, in tails.  16 blocks of 512 x 1536 with D = 256: 4 groups of 384 tails, 256 workgroups.
    // kHead 1, 2, 3, 4, 6 choose differently for few shapes; us with the pieces' sums: 8 blocks of 200 x 1000, D = 256: 57, 56,
    // 59, 60, 60; 32 of 200 x 512, D = 100: 57, 57, 59, 59, 59; 16 of 200 x 256, D = 256: 38, 35, 35, 35, 35; 10 of
    // 130 x 960, D = 128: 34, 33, 33, 35, 35; 8 of 1000 x 256, D = 64: 31, 31, 31, 31, 33.
    constexpr int kHead = 2;
    const int base = sh.S * ((sh.Dp + 63) / 64);
    L1Split k = {};
    int64_t least = INT64_MAX;
    for (int size = L1P_MAX_T; size >= 64; size -= 32) {
        const int tails = (sh.T + size - 1) / size, heads = std::max(1, std::min(256 / (base * tails), sh.B / 32));
        const int h_size = ((sh.B + heads - 1) / heads + L1P_CB - 1) / L1P_CB * L1P_CB;
        const int per_wave = std::min(size, (sh.T + 31) / 32 * 32) / L1P_WAVES;
        const int64_t cost = (int64_t)((base * tails * heads + 255) / 256) * h_size * (per_wave + kHead);
        if (cost < least) { least = cost; k.heads = heads; k.tails = tails; }
    }
    return k;
}
size_t score_bwd_pieces(const ScoreShape& sh) {
    if (sh.dist_fn != DIST_L1 || sh.score_fn == SCORE_DISTMULT || !sh.use_mfma) return 0;
    const L1Split k = l1_pair_split(sh);
    return ((k.tails > 1 ? (size_t)k.tails * sh.S * sh.B : 0) + (k.heads > 1 ? (size_t)k.heads * sh.S * sh.T : 0)) * sh.Dp;
}

template <bool FULL>
__global__ __launch_bounds__(1024) void k_score_bwd_l1_pair(const float* __restrict__ operands,
                                                            const float* __restrict__ coef,
                                                            float* __restrict__ grad_heads, float* __restrict__ grad_tails,
                                                            int S, int B, int T, int Dp, int a_c0, int b_c0,
                                                            int h_groups, int t_groups, int h_size,
                                                            const uint32_t* __restrict__ tcount) {
    __shared__ __attribute__((aligned(16))) L1PairLds lds;
    const TileId tile = xcd_tile((Dp + 63) / 64, h_groups * t_groups, S);
    const int d = tile.z, lane = threadIdx.x & 63, k = tile.x * 64 + lane;
    const int hg = tile.y / t_groups, tg = tile.y - hg * t_groups;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // merged tails: the block's distinct tails alone.  The columns between them and the forward
    // pass's limit stand for no tail position: their coefficients are zero and nothing reads
    // their gradient rows.  The groups share the live tails evenly, in steps of 32 (an even number
    // per wave: 331 instead of 343 columns per block on average on the 22.8M-row workload).
    const int live = tcount ? min(T, (int)tcount[d]) : T;
    const int t_size = ((live + t_groups - 1) / t_groups + 31) & ~31;
    const int t0 = tg * t_size, h0 = hg * h_size;
    L1Pair q;
    q.n_tail = __builtin_amdgcn_readfirstlane(min(t_size, live - t0));
    q.n_head = __builtin_amdgcn_readfirstlane(min(h_size, B - h0));
    q.col = FULL || k < Dp;
    q.k0 = tile.x * 64;
    q.kc = FULL ? k : min(k, Dp - 1);
    q.Dp = Dp; q.ldc = T;
    q.grad_a = grad_heads + ((size_t)(t_groups > 1 ? tg : 0) * S * B + (size_t)d * B + h0) * Dp;
    q.grad_b = grad_tails + ((size_t)(h_groups > 1 ? hg : 0) * S * T + (size_t)d * T + t0) * Dp;
    if (q.n_head <= 0 || q.n_tail <= 0) {  // rounding left this group empty: its pieces of the sums are zero
        if (q.col) {
            for (int b = w; b < q.n_head; b += L1P_WAVES) q.grad_a[(size_t)b * Dp + q.kc] = 0.f;
            for (int t = w; t < q.n_tail; t += L1P_WAVES) q.grad_b[(size_t)t * Dp + q.kc] = 0.f;
        }
        return;
    }
    q.a_rows = operands + (size_t)(a_c0 + d * B + h0) * Dp;
    q.b_rows = operands + (size_t)(b_c0 + d * T + t0) * Dp;
    q.coef = coef + ((size_t)d * B + h0) * T + t0;
    const int tw = ((q.n_tail + 31) & ~31) / L1P_WAVES;
#define KGE_L1P(TW_) \
    case TW_: l1_pair_wave<TW_, FULL>(q, w, lane, lds); break;
    switch (tw) {  // one of sixteen copies of the loop, chosen per group
        KGE_L1P(2) KGE_L1P(4) KGE_L1P(6) KGE_L1P(8) KGE_L1P(10) KGE_L1P(12) KGE_L1P(14) KGE_L1P(16)
        KGE_L1P(18) KGE_L1P(20) KGE_L1P(22) KGE_L1P(24) KGE_L1P(26) KGE_L1P(28) KGE_L1P(30) KGE_L1P(32)
    }
#undef KGE_L1P
}

// The pieces of the split sides added up, in group order: one wave per row of 256 columns.
__global__ __launch_bounds__(256) void k_l1_pair_sum(const float* __restrict__ head_pieces, int n_head_pieces,
                                                     const float* __restrict__ tail_pieces, int n_tail_pieces,
                                                     float* __restrict__ grad, int n_head, int n_tail, int T, int Dp,
                                                     const uint32_t* __restrict__ tcount) {
    const int slabs = (Dp + 255) / 256;
    const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int row0 = g / slabs, k = (g - row0 * slabs) * 256 + (threadIdx.x & 63) * 4;
    const int first = n_head_pieces > 1 ? 0 : n_head;  // rows of `grad` that come in pieces: [first, ..)
    const int r = first + row0;
    if (r >= n_head + (n_tail_pieces > 1 ? n_tail : 0) || k >= Dp) return;
    const bool tail = r >= n_head;
    const int q = tail ? r - n_head : r;
    if (tail && tcount && q % T >= (int)tcount[q / T]) return;  // never written, never read
    const float* src = (tail ? tail_pieces : head_pieces) + (size_t)q * Dp + k;
    const int n = tail ? n_tail_pieces : n_head_pieces;
    const size_t pitch = (size_t)(tail ? n_tail : n_head) * Dp;
    float4 sum = *reinterpret_cast<const float4*>(src);
    for (int i = 1; i < n; ++i) sum = f4add(sum, *reinterpret_cast<const float4*>(src + i * pitch));
    *reinterpret_cast<float4*>(grad + (size_t)r * Dp + k) = sum;
}

static void launch_l1_pair(const ScoreShape& sh, const float* ops, const float* coef, float* grad, float* pieces,
                           hipStream_t stream) {
    const L1Split k = l1_pair_split(sh);
    const int S = sh.S, B = sh.B, T = sh.T, Dp = sh.Dp, n_head = S * B, n_tail = S * T;
    float* const heads = k.tails > 1 ? pieces : grad;
    float* const tail_pieces = pieces + (k.tails > 1 ? (size_t)k.tails * n_head * Dp : 0);
    float* const tails = k.heads > 1 ? tail_pieces : grad + (size_t)n_head * Dp;
    const int h_size = ((B + k.heads - 1) / k.heads + L1P_CB - 1) / L1P_CB * L1P_CB;
    const dim3 grid = tile_grid((Dp + 63) / 64, k.heads * k.tails, S);
    const bool full = T % 32 == 0 && B % L1P_CB == 0 && Dp % 64 == 0;
    if (full)
        hipLaunchKernelGGL(k_score_bwd_l1_pair<true>, grid, dim3(1024), 0, stream, ops, coef, heads, tails, S, B, T, Dp, 0,
                           n_head, k.heads, k.tails, h_size, sh.tcount);
    else
        hipLaunchKernelGGL(k_score_bwd_l1_pair<false>, grid, dim3(1024), 0, stream, ops, coef, heads, tails, S, B, T, Dp, 0,
                           n_head, k.heads, k.tails, h_size, sh.tcount);
    if (k.heads == 1 && k.tails == 1) return;
    const int rows = (k.tails > 1 ? n_head : 0) + (k.heads > 1 ? n_tail : 0), slabs = (Dp + 255) / 256;
    hipLaunchKernelGGL(k_l1_pair_sum, dim3((rows * slabs + 3) / 4), dim3(256), 0, stream, heads, k.tails, tails, k.heads,
                       grad, n_head, n_tail, T, Dp, sh.tcount);
}

void launch_score_bwd(const ScoreShape& sh, const RowSource& ent, const float* rel,
                      const uint32_t* crel, const float* coef, const uint32_t* nearflag, float* grad,
                      float* pieces, hipStream_t stream) {
    BwdParams p;
    p.ent_a = ent; p.ent_b = ent; p.rel = rel; p.crel = crel; p.coef = coef; p.grad = grad;
    p.coef_div = nullptr; p.add_base = nullptr;
    p.S = sh.S; p.B = sh.B; p.T = sh.T; p.Dp = sh.Dp; p.vec_out = 1; p.use_mfma = sh.use_mfma;
    p.nearflag = nearflag;
    p.tcount = sh.tcount; p.tpad = sh.tpad;
    p.a_rel_mode = sh.operands_dense ? 0 : (sh.score_fn == SCORE_DISTMULT ? 2 : 1);
    p.a_c0 = 0; p.b_c0 = sh.S * sh.B;
    const int dist_fn = sh.score_fn == SCORE_DISTMULT ? DIST_DOT : sh.dist_fn;
    // matrix-core path: both sides in one launch (tile-aligned shapes)
    const bool plain = ent.etype == ET_F32 && !ent.index && p.a_rel_mode == 0 && ent.vec;
    const bool both = sh.use_mfma && plain && sh.B % BM_TI == 0 && sh.T % BM_TI == 0 && sh.Dp % BM_TK == 0 &&
                      (dist_fn == DIST_DOT || (dist_fn == DIST_L2 && nearflag));
    if (both) {
        const dim3 grid = tile_grid(sh.Dp / BM_TK, sh.B / BM_TI + sh.T / BM_TI, sh.S);
        // eight waves per workgroup (two per SIMD): measured faster than four at
        // every benchmark shape, few workgroups (1M-row workload) or many (22.8M-row workload)
        // three-piece bfloat16 products where the forward pass uses them (a step's L2 does not come here then:
        // split_scoring); whole slabs of 32 rows of `other` on either side (the merged tails' live counts are multiples of tpad)
        const bool split = sh.use_mfma == 2 && dist_fn == DIST_DOT && (!sh.tcount || sh.tpad % (2 * BS_KJ) == 0);
        if (split)
            hipLaunchKernelGGL(k_score_bwd_split_both, grid, dim3(512), 0, stream, p);
        else if (dist_fn == DIST_L2)
            hipLaunchKernelGGL((k_score_bwd_mfma_both<DIST_L2, 32, true, 8>), grid, dim3(512), 0, stream, p);
        else
            hipLaunchKernelGGL((k_score_bwd_mfma_both<DIST_DOT, 32, true, 8>), grid, dim3(512), 0, stream, p);
        return;
    }
    if (dist_fn == DIST_L1 && sh.use_mfma && sh.operands_dense && plain && ent.pitch == (int64_t)sh.Dp * 4 && (pieces || !score_bwd_pieces(sh))) {
        launch_l1_pair(sh, reinterpret_cast<const float*>(ent.base), coef, grad, pieces, stream);
        return;
    }
    p.side_b = 0; p.grad_c0 = p.a_c0;
    launch_bwd(p, dist_fn, stream);
    p.side_b = 1; p.grad_c0 = p.b_c0;
    launch_bwd(p, dist_fn, stream);
}


static RowSource plain_rows_bwd(const float* ptr, int D) {
    RowSource s;
    s.base = reinterpret_cast<const char*>(ptr); s.pitch = (int64_t)D * 4; s.etype = ET_F32; s.index = nullptr;
    s.count = D; s.vec = (D % 4 == 0) && ((uintptr_t)ptr % 16 == 0);
    return s;
}

// g [M, N]; dist [M, N] (L2 only, else null): gradient of the first operand
void launch_distance_grad(int dist_fn, const float* a, const float* b, const float* dist,
                          const float* g, float* grad, int M, int N, int D, hipStream_t stream) {
    BwdParams p;
    p.ent_a = plain_rows_bwd(a, D); p.ent_b = plain_rows_bwd(b, D);
    p.rel = nullptr; p.crel = nullptr;
    p.coef = g;
    p.coef_div = dist_fn == DIST_L2 ? dist : nullptr;
    p.grad = grad;
    p.S = 1; p.B = M; p.T = N; p.Dp = D;
    p.side_b = 0; p.a_rel_mode = 0;
    p.a_c0 = 0; p.b_c0 = 0; p.grad_c0 = 0; p.use_mfma = 1; p.nearflag = nullptr;
    p.tcount = nullptr; p.tpad = 1;
    p.vec_out = (D % 4 == 0) && ((uintptr_t)grad % 16 == 0);
    launch_bwd(p, dist_fn, stream);
}

}  // namespace kge
