// Per-group scale/min searches of the K-quants and IQ4_XS, one lane per group.
//
// Each function keeps a whole group (16 or 32 values) in registers and walks
// the reference's sequential candidate chain for it; parallelism comes from
// running one group per lane. The candidate order, the accept tests and every
// reduction order follow the reference's eager torch path line by line (cited
// per function), so the chosen levels and scales are bit-identical to it.
#pragma once

#include "qs_device.h"
#include "qs_wave.h"

namespace qs {

// Candidate numerators. Computed on the host in f32 exactly as the reference's
// numpy f32 chains (kq_common.py:21-30, qx_common.py:20-23) and passed in.
struct Steps {
    float v[40];
    int n;
};

// Result of the make_qkx2/qkx3 search: the levels are regenerated from
// (isc, mn) of the accepted candidate instead of being carried in registers.
struct QkxResult {
    float scale, the_min, isc, mn;
    bool degen;
};

// make_qkx_quants_eager kq_common.py:51-96 for one group of N values.
//
// The loop is bound by VALU issue: 16 instructions per value and candidate,
// two of them (the rounding and the clamp) at half rate, and the divisions.
// Those are a reciprocal of D shared by the scale and the min, a reciprocal
// of the accepted candidate's range mx - mn kept for the candidates that
// follow, and one quotient per candidate for its inverse scale; when a lane's
// operands leave the range in which quotient() is the IEEE division, the wave
// repeats the candidate's divisions with `/` (same bits where both are valid,
// so the choice is the wave's). issue_break() keeps the paired issue alive.
// Measured on random groups, clocks per candidate and wave on one SIMD: N = 32
// 1,797 with five `/` -> 1,395 with shared reciprocals -> 1,269 with the issue
// breaks (525 instructions at the paired rate would take 1,120); N = 16 871 ->
// 789 -> 689.
//
// LPG lanes per group (N values each): for shapes with few groups, where a wave's
// own latency is the time (the launches' rule has the figures). Every lane of
// the group holds the same sums, so takes the same decisions; all of them must
// call it.
template <int N, bool MAD, int LPG = 1>
QS_DEV QkxResult qkx_fit(const float (&x)[N], const float (&w)[N], const Steps& steps, float fmax) {
    float mn = x[0], mx = x[0];
#pragma unroll
    for (int i = 1; i < N; i++) {
        mn = fminf(mn, x[i]);
        mx = fmaxf(mx, x[i]);
    }
    mn = group_reduce<LPG>(mn, [](float u, float v) { return fminf(u, v); });
    mx = group_reduce<LPG>(mx, [](float u, float v) { return fmaxf(u, v); });
    mn = fminf(mn, 0.0f);
    const bool degen = (mx == mn);
    float t[N];
    const float sum_w = group_sum<LPG>(tree_sum(w));
#pragma unroll
    for (int i = 0; i < N; i++) t[i] = w[i] * x[i];
    const float sum_x = group_sum<LPG>(tree_sum(t));

    float den = degen ? 1.0f : mx - mn;
    const float iscale = fmax / den;
    float scale = 1.0f / iscale;
    float best_isc = iscale, best_mn = mn;
#pragma unroll
    for (int i = 0; i < N; i++) {
        float L = clampf(rintf(iscale * (x[i] - mn)), 0.0f, fmax);
        float d = scale * L;
        d = d + mn;
        d = d - x[i];
        t[i] = w[i] * (MAD ? fabsf(d) : d * d);
    }
    // a group with mx == mn accepts nothing (its D is 0 or NaN, and no error is
    // below -inf)
    float best = group_sum<LPG>(tree_sum(t));
    best = degen ? -__builtin_inff() : best;

    // A range mx - mn, a scale or a min within [LO, HI] and D within [DLO, DHI]
    // keep every division in quotient()'s range: the numerators of scale and min
    // are then at least 2^-96 and at most 2^120, the inverse scales (the candidates'
    // numerators are 0.5 .. 33) within 2^+-61. D is about the square of a group's
    // weights, so DHI takes imatrix entries of up to about 2^27 (with 2^36, entries
    // beyond 2^15 divided plainly: Q2_K 1024x2560 66 us instead of 60). Where DHI is
    // HI the compiler tests both with one compare: 3% faster with 8 values a lane
    // (Q4_K imatrix 400x2560 32.6 -> 31.5 us), but 1.5% slower with 4 (16x512 20.4 ->
    // 20.8), which keep two.
    constexpr float LO = 0x1p-36f, HI = 0x1p60f, DLO = 0x1p-60f, DHI = N == 4 ? 0x1p59f : HI;
    float y = recip(den);                     // of the current range
    // lanes whose current range needs `/` (a mask, so it stays in scalar registers)
    uint64_t far = wave_mask(!(den >= LO && den <= HI));
    // 16-value groups load each step one candidate ahead, so the scalar
    // load's latency is not waited for at the top of every candidate (Q2_K
    // 2-6% faster)
    constexpr bool AHEAD = N <= 16;
    // A wave whose rows keep leaving the range (few values that are not zero, whose
    // minimum is exactly 0; weights below about 1e-10) formed the quotients for
    // nothing, so after four such candidates it divides plainly at once. With 16
    // values a lane only, where the branches also make the other rows faster: Q2_K
    // bf16 2560x2560 with imatrix 114 -> 109 us, with nine tenths of the values zero
    // 135 -> 120 (125 with plain divisions only). With 4 values a lane they cost 5%
    // (16x2560 22.9 -> 24.6), with 32 1% (Q4_K imatrix 2560x2560 113.7 -> 115.2).
    constexpr bool STICKY = N == 16;
    int outs = 0;
    float step_next = steps.v[0];
#pragma unroll 1
    for (int s = 0; s < steps.n; s++) {
        const float step = AHEAD ? step_next : steps.v[s];
        if constexpr (AHEAD) step_next = steps.v[s + 1 < 40 ? s + 1 : 39];
        const bool plain = STICKY && outs >= 4;
        float isc;
        if (STICKY && (plain || far != 0)) {
            isc = step / den;
        } else {
            isc = quotient(step, den, y);
            if (!STICKY && far != 0) isc = step / den;
        }
        // the three tree sums are formed 8 values at a time (the tree over N
        // is the trees over its 8-value blocks, then the tree over the block
        // sums), so only one block of products is live at once
        constexpr int B = N < 8 ? N : 8, NB = N / B;
        float La[N], sa[NB], sb[NB], sc[NB];
#pragma unroll
        for (int k = 0; k < NB; k++) {
            float a[B], b[B], c[B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int i = B * k + j;
                La[i] = clampf(rintf(isc * (x[i] - mn)), 0.0f, fmax);
                a[j] = w[i] * La[i];
                b[j] = a[j] * La[i];
                c[j] = a[j] * x[i];
            }
            issue_break(a[3]);
            sa[k] = tree_sum(a);
            sb[k] = tree_sum(b);
            sc[k] = tree_sum(c);
            issue_break(sc[k]);
        }
        const float sum_l = group_sum<LPG>(tree_sum(sa)), sum_l2 = group_sum<LPG>(tree_sum(sb)),
                    sum_xl = group_sum<LPG>(tree_sum(sc));
        const float D = sum_w * sum_l2 - sum_l * sum_l;
        const float Dsafe = D > 0 ? D : 1.0f;
        const float num_s = sum_w * sum_xl - sum_x * sum_l, num_m = sum_l2 * sum_x - sum_l * sum_xl;
        // only a candidate that can be accepted has to be exact
        const bool live = D > 0;
        float this_scale, this_min, den_acc;
        bool out = live;
        if (!plain) {
            const float yd = recip(Dsafe);
            this_scale = quotient(num_s, Dsafe, yd);
            this_min = quotient(num_m, Dsafe, yd);
            const float q_s = fabsf(this_scale), q_m = fabsf(this_min);
            if (this_min > 0) {
                this_scale = sum_xl / fmaxf(sum_l2, F32_TINY);
                this_min = 0.0f;
            }
            den_acc = mx - this_min;
            // q_hi keeps a NaN (v_maximum3_f32; a quotient of an overflowed numerator,
            // where `/` gives an infinity), which then fails the test; fminf drops it
            const float q_lo = fminf(fminf(q_s, q_m), den_acc);
            const float q_hi = __builtin_elementwise_maximum(__builtin_elementwise_maximum(q_s, q_m), den_acc);
            out = live && !(q_lo >= LO && q_hi <= HI && D >= DLO && D <= DHI);
        }
        if (plain || wave_any(out)) {
            outs++;
            this_scale = num_s / Dsafe;
            this_min = num_m / Dsafe;
            if (this_min > 0) {
                this_scale = sum_xl / fmaxf(sum_l2, F32_TINY);
                this_min = 0.0f;
            }
            den_acc = mx - this_min;
        }
        const float y_acc = recip(den_acc);
        float se[NB];
#pragma unroll
        for (int k = 0; k < NB; k++) {
            float e8[B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int i = B * k + j;
                float d = this_scale * La[i];
                d = d + this_min;
                d = d - x[i];
                e8[j] = w[i] * (MAD ? fabsf(d) : d * d);
            }
            issue_break(e8[3]);
            se[k] = tree_sum(e8);
            issue_break(se[k]);
        }
        const float cur = group_sum<LPG>(tree_sum(se));
        const bool accept = live && cur < best;
        const uint64_t acc = wave_mask(accept);
        far = (far & ~acc) | (wave_mask(out) & acc);
        if (accept) {
            best_isc = isc;
            best_mn = mn;
            scale = this_scale;
            mn = this_min;
            best = cur;
            den = den_acc;
            y = y_acc;
        }
    }
    QkxResult r;
    r.scale = degen ? 0.0f : scale;
    r.the_min = (mn == 0.0f) ? 0.0f : -mn;
    r.isc = best_isc;
    r.mn = best_mn;
    r.degen = degen;
    return r;
}

// level i of the accepted make_qkx candidate
QS_DEV float qkx_level(const QkxResult& r, float x, float fmax) {
    return r.degen ? 0.0f : clampf(rintf(r.isc * (x - r.mn)), 0.0f, fmax);
}

// Final levels of a group: clamp(rint(t[i] / d), lo, hi) for the N values of one
// divisor, from one reciprocal (5 full-rate instructions a value for the
// division instead of 10 at mostly half rate). The rounded quotient is IEEE's
// where |t| >= 2^-96; below that, with |d| >= 2^-36, both quotients round to
// zero. Waves holding a divisor or value outside the range divide with `/`.
// Lanes with d = 0 get no meaningful levels.
template <int N>
QS_DEV void quotient_levels(const float (&t)[N], float d, float lo, float hi, float (&v)[N]) {
    const float y = recip(d);
    float m = fabsf(t[0]);
#pragma unroll
    for (int i = 0; i < N; i++) {
        m = fmaxf(m, fabsf(t[i]));
        v[i] = clampf(rintf(quotient(t[i], d, y)), lo, hi);
        if (i % 4 == 3) issue_break(v[i]);
    }
    const float ad = fabsf(d);
    const bool in = m <= 0x1p60f && ad >= 0x1p-36f && ad <= 0x1p36f;
    if (wave_any(!in && d != 0.0f)) {
#pragma unroll
        for (int i = 0; i < N; i++) v[i] = clampf(rintf(t[i] / d), lo, hi);
    }
}

// N levels (integers 0 .. 255) as bytes to N consecutive bytes of LDS at a
// boundary of min(N, 16) bytes: one conversion and merge per value, 16-byte stores (one
// byte store per value took a quarter of the requantization)
template <int N>
QS_DEV void store_levels(const float (&v)[N], uint8_t* o) {
    uint32_t w[N / 4];
#pragma unroll
    for (int j = 0; j < N / 4; j++) {
        w[j] = 0;
#pragma unroll
        for (int b = 0; b < 4; b++) w[j] = __builtin_amdgcn_cvt_pk_u8_f32(v[4 * j + b], b, w[j]);
    }
    if constexpr (N >= 16) {
#pragma unroll
        for (int q = 0; q < N / 16; q++)
            reinterpret_cast<u32x4*>(o)[q] = u32x4{w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]};
    } else {
#pragma unroll
        for (int j = 0; j < N / 4; j++) reinterpret_cast<uint32_t*>(o)[j] = w[j];
    }
}

// make_qp_quants_eager kq_common.py:99-141, in three parts: qp_trial (one
// trial's weighted error), qp_finish (levels, sums and refinement passes for
// the chosen iscale) and the choice between them, made by qp_fit on one lane
// or by qp_fit_spread over several.

// The weighted error of the levels rint(isc * x), clamped to fmax unless
// `clamp` is false: the first pass (kq_common.py:107-109) does not clamp.
template <int N>
QS_DEV float qp_trial(const float (&x)[N], const float (&w)[N], float isc, float fmax, bool clamp) {
    const float r = 1.0f / isc;
    return cascade8_of<N>([&](int i) {
        float l = rintf(isc * x[i]);
        l = clamp ? fminf(l, fmax) : l;
        float d = x[i] - r * l;
        return w[i] * (d * d);
    });
}

// kq_common.py:118-141 for the chosen iscale: writes the levels to L and
// returns the scale.
template <int N>
QS_DEV float qp_finish(const float (&x)[N], const float (&w)[N], float fmax, float iscale, bool dead,
                       float (&L)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) L[i] = fminf(rintf(iscale * x[i]), fmax);
    float sumlx = cascade8_of<N>([&](int i) { return (w[i] * x[i]) * L[i]; });
    float suml2 = cascade8_of<N>([&](int i) { return (w[i] * L[i]) * L[i]; });
#pragma unroll 1
    for (int pass = 0; pass < 5; pass++) {
        bool changed = false;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const float xi = x[i], Li = L[i];
            float wi = w[i];
            // keeps wi * xi inside the pass: hoisting the N products out of
            // the loop would hold N more registers for the whole fit
            keep_in_register(wi);
            const float slx = sumlx - (wi * xi) * Li;
            const float sl2 = suml2 - (wi * Li) * Li;
            const bool ok = slx > 0 && sl2 > 0;
            const float newl = fminf(rintf((xi * sl2) / (ok ? slx : 1.0f)), fmax);
            const float slx2 = slx + (wi * xi) * newl;
            const float sl22 = sl2 + (wi * newl) * newl;
            if (ok && newl != Li && (slx2 * slx2) * suml2 > (sumlx * sumlx) * sl22) {
                L[i] = newl;
                sumlx = slx2;
                suml2 = sl22;
                changed = true;
            }
        }
        // a pass that commits nothing leaves L, sumlx and suml2 as they were,
        // so every later pass repeats it (the C loop's early break, which the
        // reference's five passes stand for, kq_common.py:121-136): the wave stops
        // once none of its lanes committed
        if (!wave_any(changed)) break;
    }
    float scale = suml2 > 0 ? sumlx / fmaxf(suml2, F32_TINY) : 0.0f;
    if (dead) {
        scale = 0.0f;
#pragma unroll
        for (int i = 0; i < N; i++) L[i] = 0.0f;
    }
    return scale;
}


template <int N>
QS_DEV float qp_max(const float (&x)[N]) {
    float mx = x[0];
#pragma unroll
    for (int i = 1; i < N; i++) mx = fmaxf(mx, x[i]);
    return mx;
}

// make_qp_quants_eager on one lane (N = 8, 16, 32). Writes the levels to L
// and returns the scale.
template <int N>
QS_DEV float qp_fit(const float (&x)[N], const float (&w)[N], int nmax, const float (&steps)[8], float (&L)[N]) {
    const float fmax = (float)nmax;
    const float mx = qp_max(x);
    const bool dead = mx < GROUP_MAX_EPS;
    const float mxs = dead ? 1.0f : mx;

    float iscale = rdiv(fmax, mxs);
    float best_mse = qp_trial<N>(x, w, iscale, fmax, false);
#pragma unroll 1
    for (int s = 0; s < 8; s++) {
        const float isc = rdiv(steps[s], mxs);
        const float mse = qp_trial<N>(x, w, isc, fmax, true);
        if (mse < best_mse) {
            best_mse = mse;
            iscale = isc;
        }
    }
    return qp_finish<N>(x, w, fmax, iscale, dead, L);
}

// make_qp_quants_eager for one superblock's N sub-block scales (or mins),
// spread over P consecutive lanes (c = 0..P-1) that all hold x and w. The
// nine trials (the first pass, then the eight candidates) do not depend on
// each other, only the choice among them does, so lane c runs trials c,
// c + P, ...; their (error, iscale) pairs meet in xch (18 floats of LDS) and
// every lane makes the reference's choice in trial order (the first strict
// minimum) and finishes the fit. Every lane of the wave must call it (it
// holds a wave barrier); all P lanes return the same scale and levels.
template <int N, int P, bool WL = false>
QS_DEV float qp_fit_spread(const float (&x)[N], const float (&w)[N], int nmax, const float (&steps)[8],
                           float (&L)[N], int c, float* xch) {
    static_assert(P >= 1, "lanes past the ninth hold no trial");
    const float fmax = (float)nmax;
    const float mx = qp_max(x);
    const bool dead = mx < GROUP_MAX_EPS;
    const float mxs = dead ? 1.0f : mx;
#pragma unroll
    for (int k = 0; k < (9 + P - 1) / P; k++) {
        const int e = c + k * P;
        if (e < 9) {
            float num = fmax;        // trial 0: nmax / max; trial e: candidate e - 1
#pragma unroll
            for (int j = 0; j < 8; j++) num = e == j + 1 ? steps[j] : num;
            const float isc = rdiv(num, mxs);
            xch[2 * e] = qp_trial<N>(x, w, isc, fmax, e != 0);
            xch[2 * e + 1] = isc;
        }
    }
    wave_sync<WL>();
    float best_mse = xch[0], iscale = xch[1];
#pragma unroll
    for (int e = 1; e < 9; e++) {
        const float mse = xch[2 * e];
        if (mse < best_mse) {
            best_mse = mse;
            iscale = xch[2 * e + 1];
        }
    }
    return qp_finish<N>(x, w, fmax, iscale, dead, L);
}

// make_qx_quants_eager qx_common.py:52-82 for one group of 16 values.
// Returns the scale; the levels are regenerated from (isc) by qx_level.
struct QxResult {
    float scale, isc;
    bool live;
};

// sums of one make_qx trial: the levels clamp(rint(isc * x), -nmax, nmax - 1)
// and their seq-sums sum w x L, sum w L^2 (qx_common.py:61-63, :68-70)
template <int N>
QS_DEV float2 qx_trial(const float (&x)[N], const float (&w)[N], float isc, float fmax) {
    float t[N], u[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        float La = clampf(rintf(isc * x[i]), -fmax, fmax - 1.0f);
        t[i] = (w[i] * x[i]) * La;
        u[i] = (w[i] * La) * La;
    }
    float st = t[0], su = u[0];
#pragma unroll
    for (int i = 1; i < N; i++) {
        st = st + t[i];
        su = su + u[i];
        if (i == N / 2) issue_break(st);
    }
    return make_float2(st, su);
}

template <int N>
QS_DEV QxResult qx_fit(const float (&x)[N], const float (&w)[N], int nmax, const Steps& steps) {
    const float fmax = (float)nmax;
    float amax;
    const float mx = absmax_first(x, amax);
    const bool live = amax >= GROUP_MAX_EPS;
    const float mxs = live ? mx : 1.0f;
    const float iscale = rdiv(-fmax, mxs);
    const float2 s0 = qx_trial<N>(x, w, iscale, fmax);
    const float sumlx = s0.x, suml2 = s0.y;
    float scale = suml2 != 0 ? sumlx / suml2 : 0.0f;
    float best = scale * sumlx, best_isc = iscale;
    float step_next = steps.v[0];      // loaded one candidate ahead (Q3_K 4%, Q6_K 2% faster)
#pragma unroll 1
    for (int s = 0; s < steps.n; s++) {
        const float step = step_next;
        step_next = steps.v[s + 1 < 40 ? s + 1 : 39];
        const float isc = rdiv(-step, mxs);
        const float2 sc = qx_trial<N>(x, w, isc, fmax);
        const float slx = sc.x, sl2 = sc.y;
        if (sl2 > 0 && slx * slx > best * sl2) {
            const float cand = slx / sl2;
            scale = cand;
            best = cand * slx;
            best_isc = isc;
        }
    }
    QxResult r;
    r.scale = live ? scale : 0.0f;
    r.isc = best_isc;
    r.live = live;
    return r;
}

// floats of LDS a 19-trial make_qx (qx_fit_spread, NS = 18) and a 16-trial IQ4
// search exchange per group, odd so that groups start in different banks
constexpr int QX_XCH = 3 * 19, IQ4_XCH = 33;

// make_qx_quants_eager for one superblock's N sub-block scales, spread over
// P consecutive lanes (c = 0..P-1) that all hold x and w, for NS candidates
// (the host's steps.n). A trial's levels and sums depend only on its iscale,
// not on earlier accepts, so lane c forms the sums of trials c, c + P, ...
// (trial 0: the first pass; trial e: candidate e - 1); they meet in xch
// (3 (NS + 1) floats of LDS) and every lane runs the accept chain in
// candidate order. Every lane of the wave must call it (it holds a wave
// barrier); all P lanes return the same result.
template <int N, int P, int NS, bool WL = false>
QS_DEV QxResult qx_fit_spread(const float (&x)[N], const float (&w)[N], int nmax, const Steps& steps,
                              int c, float* xch) {
    const float fmax = (float)nmax;
    float amax;
    const float mx = absmax_first(x, amax);
    const bool live = amax >= GROUP_MAX_EPS;
    const float mxs = live ? mx : 1.0f;
#pragma unroll
    for (int k = 0; k < (NS + 1 + P - 1) / P; k++) {
        const int e = c + k * P;
        if (e <= NS) {
            float num = fmax;
#pragma unroll
            for (int j = 0; j < NS; j++) num = e == j + 1 ? steps.v[j] : num;
            const float isc = rdiv(-num, mxs);
            const float2 sc = qx_trial<N>(x, w, isc, fmax);
            xch[3 * e] = sc.x;
            xch[3 * e + 1] = sc.y;
            xch[3 * e + 2] = isc;
        }
    }
    wave_sync<WL>();
    const float sumlx = xch[0], suml2 = xch[1];
    float scale = suml2 != 0 ? sumlx / suml2 : 0.0f;
    float best = scale * sumlx, best_isc = xch[2];
#pragma unroll 1
    for (int e = 1; e <= NS; e++) {
        const float slx = xch[3 * e], sl2 = xch[3 * e + 1];
        if (sl2 > 0 && slx * slx > best * sl2) {
            const float cand = slx / sl2;
            scale = cand;
            best = cand * slx;
            best_isc = xch[3 * e + 2];
        }
    }
    QxResult r;
    r.scale = live ? scale : 0.0f;
    r.isc = best_isc;
    r.live = live;
    return r;
}

// level (0 .. 2*nmax-1) of the accepted make_qx candidate
QS_DEV float qx_level(const QxResult& r, float x, float fmax) {
    return r.live ? clampf(rintf(r.isc * x), -fmax, fmax - 1.0f) + fmax : 0.0f;
}

// make_q3_quants_eager qx_common.py:85-121 for one group of 16 (w = x*x).
// Writes levels (0 .. 2*nmax-1) and returns the scale.
template <int N>
QS_DEV float q3_fit(const float (&x)[N], int nmax, float (&L)[N]) {
    const float fmax = (float)nmax;
    float w[N], t[N], u[N];
#pragma unroll
    for (int i = 0; i < N; i++) w[i] = x[i] * x[i];
    float amax;
    const float mx = absmax_first(x, amax);
    const bool live = amax >= GROUP_MAX_EPS;
    const float mxs = live ? mx : 1.0f;
    const float iscale = rdiv(-fmax, mxs);
#pragma unroll
    for (int i = 0; i < N; i++) {
        L[i] = clampf(rintf(iscale * x[i]), -fmax, fmax - 1.0f);
        t[i] = (w[i] * x[i]) * L[i];
        u[i] = (w[i] * L[i]) * L[i];
    }
    float sumlx = seq_sum(t), suml2 = seq_sum(u);
#pragma unroll 1
    for (int pass = 0; pass < 5; pass++) {
        bool changed = false;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const float xi = x[i], wi = w[i], Li = L[i];
            const float slx = sumlx - (wi * xi) * Li;
            const bool ok = slx > 0;
            const float sl2 = suml2 - (wi * Li) * Li;
            const float newl = clampf(rintf((xi * sl2) / (ok ? slx : 1.0f)), -fmax, fmax - 1.0f);
            const float slx2 = slx + (wi * xi) * newl;
            const float sl22 = sl2 + (wi * newl) * newl;
            if (ok && newl != Li && sl22 > 0 && (slx2 * slx2) * suml2 > (sumlx * sumlx) * sl22) {
                L[i] = newl;
                sumlx = slx2;
                suml2 = sl22;
                changed = true;
            }
        }
        if (!wave_any(changed)) break;        // as in qp_fit (qx_common.py:100-114)
    }
    const float scale = suml2 > 0 ? sumlx / suml2 : 0.0f;
#pragma unroll
    for (int i = 0; i < N; i++) L[i] = live ? L[i] + fmax : 0.0f;
    return live ? scale : 0.0f;
}

// ---- IQ4_XS (iq4_xs.py:23-76) ----

// _best_index (iq4_xs.py:35-39) as a table over floor(2 al): the bracket's
// compare `al - lo < hi - al` is `al < (lo + hi) / 2` (near a midpoint both
// differences are exact), and the midpoints of the integer LUT are multiples
// of one half, so the projection only changes where 2 al is an integer. Entry
// e stands for floor(2 al) = e (e < 512) or e - 1024 (the negative half): a
// masked floor is always inside the table. `val` holds the LUT value, `idx`
// its index, one byte each: a search's lookups then fall into the ~60 words
// around zero, about one per LDS bank.
// Measured (IQ4_XS with imatrix, bf16 9728x2560): the bracket pair read as
// float2 at clamp(floor(al)) + 128 and compared took 14 VALU instructions per
// value and trial and two LDS words, this takes 9 and a byte.
struct Iq4Tab {
    alignas(16) int8_t val[1024];
    alignas(16) uint8_t idx[1024];
};

constexpr Iq4Tab iq4_make_tab() {
    constexpr int V[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
    Iq4Tab t{};
    for (int e = 0; e < 1024; e++) {
        const int k = e < 512 ? e : e - 1024;
        int i = 0;
        while (i < 15 && V[i] + V[i + 1] <= k) i++;
        t.val[e] = (int8_t)V[i];
        t.idx[e] = (uint8_t)i;
    }
    return t;
}

static __device__ const Iq4Tab iq4_tab_const = iq4_make_tab();

// a one-wave workgroup's copy of the table in LDS (16 bytes per lane and half)
QS_DEV void iq4_load_tab(Iq4Tab& t) {
    const int lane = (int)threadIdx.x;
    reinterpret_cast<u32x4*>(t.val)[lane] = reinterpret_cast<const u32x4*>(iq4_tab_const.val)[lane];
    reinterpret_cast<u32x4*>(t.idx)[lane] = reinterpret_cast<const u32x4*>(iq4_tab_const.idx)[lane];
}

// floor(v) as an integer, saturating, 0 for NaN (v_cvt_flr_i32_f32)
QS_DEV int floor_int(float v) {
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(v));     // the compiler takes two instructions
    return r;
}

// LUT value of _best_index(al) from al2 = 2 al, for |al| < 256 (a trial's
// |al| is at most 134). NaN takes entry 0: the sums it enters are NaN or
// infinite whatever the value.
QS_DEV float iq4_project(float al2, const Iq4Tab& t) { return (float)t.val[floor_int(al2) & 1023]; }

// LUT index of _best_index(al) for any al; NaN takes index 1, as the bracket
// compare does
QS_DEV int iq4_project_index(float al, const Iq4Tab& t) {
    const float v = al == al ? clampf(2.0f * al, -512.0f, 511.0f) : -200.0f;    // -200: index 1
    return t.idx[floor_int(v) & 1023];
}

// qs of one block of 32 (iq4_xs.py:180-186): byte j holds the indices of
// values j and j + 16, so a lane packs its own block in registers
QS_DEV void iq4_pack(const float (&x)[32], float id, const Iq4Tab& t, uint32_t (&w)[4]) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            lo |= (uint32_t)iq4_project_index(id * x[4 * k + b], t) << (8 * b);
            hi |= (uint32_t)iq4_project_index(id * x[4 * k + b + 16], t) << (8 * b);
        }
        w[k] = lo | (hi << 4);
    }
}

// _search_scales_eager iq4_xs.py:52-76 for one block of 32. The two sums of
// a candidate run left to right (seq_sum's order) over terms staged CH values
// at a time: the imatrix kernels hold 128 VGPRs with CH = 16, a fourth wave per
// SIMD (6-7% faster; IQ4_XS at one lane per block spills 8, 14 with the AMD host's
// maps). The kernels without imatrix hold 81-106 with all 32 staged (CH = 32), four
// waves as well.
// LPG > 1: the LPG lanes c = 0 .. LPG - 1 of a block all hold it, lane c forms the
// sums of trials c, c + LPG, ... (a trial does not depend on earlier accepts),
// they meet in xch (32 floats of LDS), and every lane runs the accept chain in
// trial order.
template <int CH, int LPG>
QS_DEV float iq4_scale_search(const float (&x)[32], const float (&w)[32], const Iq4Tab& tab, int c0, float* xch) {
    float amax;
    const float mx = absmax_first(x, amax);
    const bool live = fabsf(mx) >= GROUP_MAX_EPS;
    const float mxs = live ? mx : 1.0f;
    const float d0 = -mxs / -127.0f;
    const float id0 = 1.0f / d0;
    auto sums = [&](float iv, float& sqx, float& sq2) {
        const float iv2 = 2.0f * iv;      // 2 fl(iv x) = fl(2 iv x)
#pragma unroll
        for (int c = 0; c < 32; c += CH) {
            float t[CH], u[CH];
#pragma unroll
            for (int i = 0; i < CH; i++) {
                const float q = iq4_project(iv2 * x[c + i], tab);
                const float wq = w[c + i] * q;
                t[i] = wq * x[c + i];
                u[i] = wq * q;
            }
#pragma unroll
            for (int i = 0; i < CH; i++) {
                sqx = c + i == 0 ? t[i] : sqx + t[i];
                sq2 = c + i == 0 ? u[i] : sq2 + u[i];
            }
        }
    };
    float sumqx, sumq2;
    if constexpr (LPG > 1) {
#pragma unroll 1
        for (int e = c0; e < 16; e += LPG) {
            sums(e == 0 ? id0 : rdiv((float)(e - 8 - 127), mxs), sumqx, sumq2);
            xch[2 * e] = sumqx;
            xch[2 * e + 1] = sumq2;
        }
        wave_sync();
        sumqx = xch[0];
        sumq2 = xch[1];
    } else {
        sums(id0, sumqx, sumq2);
    }
    float d = sumq2 > 0 ? sumqx / sumq2 : 0.0f;
    float best = d * sumqx;
#pragma unroll 1
    for (int itry = -7; itry <= 7; itry++) {
        if constexpr (LPG > 1) {
            sumqx = xch[2 * (itry + 8)];
            sumq2 = xch[2 * (itry + 8) + 1];
        } else {
            sums(rdiv((float)(itry - 127), mxs), sumqx, sumq2);
        }
        if (sumq2 > 0 && sumqx * sumqx > best * sumq2) {
            const float nd = sumqx / sumq2;
            d = nd;
            best = nd * sumqx;
        }
    }
    return live ? d : 0.0f;
}

}  // namespace qs
