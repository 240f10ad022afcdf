// Device functions that the scoring epilogues and the row-wise loss kernels share: logSigmoid in its
// forms, a score column's loss term, and the ratios that separate cancelled pairs from the rest.
#pragma once

#include "kge_device.h"

namespace kge {

// logSigmoid and its derivative exactly as src/pag/pag.cpp:894-903
DEVINL float log_sigmoid(float z) { return z > -11.f ? -log1pf(expf(-z)) : z; }
DEVINL float log_sigmoid_grad(float z) { return 1.f / (1.f + expf(fminf(z, 11.f))); }

// The same two functions from ONE hardware exponential (the scoring epilogues
// evaluate them once per score): with u = exp(-|z|) in (0, 1],
//   z >= 0:        logsig = -log1p(u),     dlogsig = u' / (1 + u'),  u' = max(u, e^-11)  (the +11 clamp;
//                  u / (1 + u) grows with u, so the clamp can move to the quotient)
//   -11 < z < 0:   logsig = z - log1p(u),  dlogsig = 1 / (1 + u)
//   z <= -11:      logsig = z              (the reference drops the log1p term there)
// log1p(u) = log(w) - ((w - 1) - u) / w with w = 1 + u keeps the low bits of u.
DEVINL void log_sigmoid_both(float z, float& value, float& grad) {
    // single hardware instructions: exp2, rcp and log2 (about 1 ulp each; w is in [1, 2], so
    // none of the range fix-ups of the library forms is needed)
    const float u = __builtin_amdgcn_exp2f(-1.44269504089f * fabsf(z));
    const float w = 1.f + u;
    const float rw = __builtin_amdgcn_rcpf(w);
    const float l1p = 0.69314718056f * __builtin_amdgcn_logf(w) - ((w - 1.f) - u) * rw;
    // straight-line selects (lanes of a wave mix both signs of z):
    //   value = min(z, 0) - log1p(u), without the log1p term for z <= -11
    //   grad  = u / (1 + u) clamped below at its value for u = e^-11 (z >= 0), 1 / (1 + u) (z < 0)
    value = fminf(z, 0.f) - (z > -11.f ? l1p : 0.f);
    const float g_pos = fmaxf(u * rw, 1.670142184e-5f);  // e^-11 / (1 + e^-11)
    grad = z >= 0.f ? g_pos : rw;
}

// The same for both signs of one score: exp(-|s|) serves z = s and z = -s alike.
struct LogSigmoid {
    float s, rw, l1p, g_big;
    DEVINL LogSigmoid() {}
    DEVINL explicit LogSigmoid(float score) : s(score) {
        const float u = __builtin_amdgcn_exp2f(-1.44269504089f * fabsf(s));
        const float w = 1.f + u;
        rw = __builtin_amdgcn_rcpf(w);
        l1p = 0.69314718056f * __builtin_amdgcn_logf(w) - ((w - 1.f) - u) * rw;
        g_big = fmaxf(u * rw, 1.670142184e-5f);  // e^-11 / (1 + e^-11)
    }
    DEVINL float plus_value() const { return fminf(s, 0.f) - (s > -11.f ? l1p : 0.f); }
    DEVINL float minus_value() const { return fminf(-s, 0.f) - (s < 11.f ? l1p : 0.f); }
    DEVINL float plus_grad() const { return s >= 0.f ? g_big : rw; }
    DEVINL float minus_grad() const { return s <= 0.f ? g_big : rw; }
};

// The logsigmoid loss of one score column that stands for `mult` tail positions, one of them the
// positive's label if `pos` (src/poplar_kge.cpp:615-636 summed over the positions that share the
// row): returns the loss term (before the normalisation) and sets d loss / d score (times grad_scale).
DEVINL float logsigmoid_column(float score, bool pos, float mult, float w_pos, float w_neg, float grad_scale,
                               float& dscore) {
    const LogSigmoid z(score);
    const float wp = pos ? w_pos : 0.f, wn = (mult - (pos ? 1.f : 0.f)) * w_neg;
    dscore = (wn * z.minus_grad() - wp * z.plus_grad()) * grad_scale;
    return -(wp * z.plus_value() + wn * z.minus_value());
}

constexpr float kCancelRatio = 0.125f;  // recompute when d^2 < ratio * (|a|^2 + |b|^2)
// Below this ratio the backward's product form self*sum(c) - sum(c*other) would
// lose accuracy against the reference's c*(self-other); such 32x32 sub-blocks
// are flagged for the backward kernel, which handles them in the direct form.
constexpr float kNearRatio = 1.f / 4096.f;

}  // namespace kge
