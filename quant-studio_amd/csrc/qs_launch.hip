// Per-type launch geometry and template dispatch of the quantizer kernels.
// Built once per source element type (-DQS_LAUNCH_SRC=<qs::SRC_* value>), so
// the three instantiation sets compile in parallel.
#include <hip/hip_runtime.h>

#include <tuple>
#include <utility>

#include "quant_studio.h"
#include "qs_launch.h"

#ifndef QS_LAUNCH_SRC
#error "build with -DQS_LAUNCH_SRC=<source type id> (quant-studio_amd/build.py)"
#endif

namespace qs_launch {
namespace {

// Launch through hipLaunchKernel so its status comes back as the return
// value: the caller's pending hipGetLastError() state is neither read nor
// reset by this library.
template <typename... P, typename... A>
hipError_t launch(void (*kernel)(P...), dim3 grid, dim3 block, hipStream_t st, A&&... args) {
    static_assert(sizeof...(P) == sizeof...(A), "kernel argument count");
    std::tuple<P...> vals(std::forward<A>(args)...);
    void* argv[sizeof...(P)];
    std::apply([&](auto&... v) {
        int i = 0;
        ((argv[i++] = static_cast<void*>(&v)), ...);
    }, vals);
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, argv, 0, st);
}

qs::IqSteps iq_steps(float base, float delta, int lo, int hi) {
    qs::IqSteps s{};
    s.n = 0;
    for (int i = lo; i <= hi; i++) {
        float t = (float)i * delta;
        s.v[s.n++] = base + t;
    }
    return s;
}

// candidate numerators, f32 chains as kq_common.py:21-30 and qx_common.py:20-23
qs::Steps qkx_steps(float rmin, float rdelta, int nstep, int nmax) {
    qs::Steps s{};
    for (int i = 0; i <= nstep; i++) {
        float t = rdelta * (float)i;
        t = rmin + t;
        s.v[i] = t + (float)nmax;
    }
    s.n = nstep + 1;
    return s;
}

qs::QpSteps qp_steps(int nmax) {
    qs::QpSteps s{};
    int n = 0;
    for (int i = -4; i <= 4; i++) {
        if (!i) continue;
        float t = 0.1f * (float)i;
        s.v[n++] = t + (float)nmax;
    }
    return s;
}

qs::Steps qx_steps(int nmax) {
    qs::Steps s{};
    int n = 0;
    for (int i = -9; i <= 9; i++) {
        if (!i) continue;
        float t = 0.1f * (float)i;
        s.v[n++] = (float)nmax + t;
    }
    s.n = n;
    return s;
}

template <int SRC, qs::B32 T>
hipError_t launch_b32(const qs::KArgs& a, hipStream_t st) {
    const unsigned g = (unsigned)((a.n_units + qs::Q40_BLOCKS_PER_WG - 1) / qs::Q40_BLOCKS_PER_WG);
    return launch(qs::k_b32<SRC, T>, dim3(g), dim3(256), st, a);
}

// One wave per workgroup of 64 / lps superblocks
dim3 sb_grid(const qs::KArgs& a, int lps) { return dim3((unsigned)((a.n_units + 64 / lps - 1) / (64 / lps))); }

// Lanes per group of the make_qkx kernels. A launch of a wave or two per SIMD
// (256 CUs x 4) takes as long as one wave (two waves share a SIMD's issue at
// full rate), whose time is its instruction count: over 2, 4, 8 lanes a group
// takes 0.65, 0.5, 0.42 of one wave's time and 1.14, 1.5, 2.1 times the work.
// So each split is taken up to the 2 or 3 waves per SIMD where the next
// smaller one overtakes it. Measured, k = 2048 bf16, us at 1 / 2 / 4 / 8 lanes per
// group for a number of superblocks:
//   Q4_K imatrix  512 52.8 / 34.3 / 25.7 / 22.7    2,048 53.7 / 36.4 / 26.7 / 26.4
//                 6,144 54.8 / 42.8 / 41.1 / 53.0  8,192 55.6 / 43.1 / 50.7 / 66.5
//                 12,288 61.6 / 57.6 / 69.3 / 93.5 16,384 63.0 / 71.4 / 88.0 / 121
//   Q4_K          2,048 29.4 / 20.7 / 15.3 / 15.4  6,144 30.0 / 24.4 / 23.1 / 29.8
//                 12,288 34.5 / 32.3 / 38.8 / 52.0 16,384 34.9 / 39.7 / 49.1 / 66.9
//   Q5_K          2,048 23.6 / 17.0 / 13.1 / 12.9  6,144 24.3 / 20.1 / 19.0 / 24.2
//                 12,288 28.3 / 26.4 / 31.7 / 42.0 16,384 28.8 / 32.1 / 39.9 / 53.8
// and Q2_K (16 lanes per superblock at one per group) at 1 / 2 / 4:
//   with imatrix  512 37.9 / 29.9 / 25.8  2,048 41.1 / 30.8 / 29.0  4,096 40.1 / 34.7 / 42.7
//                 6,144 45.4 / 43.8 / 56.4  8,192 46.0 / 53.0 / 70.8
//   without       2,048 15.9 / 12.4 / 12.0  4,096 15.4 / 13.9 / 17.5  6,144 17.2 / 17.9 / 22.9
constexpr int64_t kSplit8 = 2048, kSplit4 = 6144, kSplit2 = 12288, kSplit2Q2 = 4096;

template <int SRC, bool IMAT, int NMAX, int SQ>
hipError_t launch_q45(const qs::KArgs& a, hipStream_t st, const qs::Steps& steps) {
    const dim3 wave(64);
    if (a.n_units <= kSplit8)
        return launch(qs::k_q45_k<SRC, IMAT, NMAX, SQ, 8>, sb_grid(a, 64), wave, st, a, steps, qp_steps(63));
    if (a.n_units <= kSplit4)
        return launch(qs::k_q45_k<SRC, IMAT, NMAX, SQ, 4>, sb_grid(a, 32), wave, st, a, steps, qp_steps(63));
    if (a.n_units <= kSplit2)
        return launch(qs::k_q45_k<SRC, IMAT, NMAX, SQ, 2>, sb_grid(a, 16), wave, st, a, steps, qp_steps(63));
    return launch(qs::k_q45_k<SRC, IMAT, NMAX, SQ, 1>, sb_grid(a, 8), wave, st, a, steps, qp_steps(63));
}

template <int SRC, bool IMAT, int SQ>
hipError_t launch_q2(const qs::KArgs& a, hipStream_t st, const qs::Steps& steps) {
    const dim3 wave(64);
    if (a.n_units <= kSplit8)
        return launch(qs::k_q2_k<SRC, IMAT, SQ, 4>, sb_grid(a, 64), wave, st, a, steps, qp_steps(15));
    if (a.n_units <= kSplit2Q2)
        return launch(qs::k_q2_k<SRC, IMAT, SQ, 2>, sb_grid(a, 32), wave, st, a, steps, qp_steps(15));
    return launch(qs::k_q2_k<SRC, IMAT, SQ, 1>, sb_grid(a, 16), wave, st, a, steps, qp_steps(15));
}

// Four lanes per group for the trials of Q3_K with an imatrix and IQ4_XS, where the
// launch has few waves (the reason is that of launch_q45; each lane repeats the
// weights and the levels, so the work grows faster). Measured, k = 2048 bf16, us at
// 1 / 4 lanes per group:
//   Q3_K imatrix    512 superblocks 14.9 / 12.6  2,048 16.0 / 13.8  3,072 15.6 / 16.6
//   IQ4_XS imatrix  512 18.5 / 12.0  4,096 20.2 / 14.3  6,144 20.3 / 17.4  10,240 23.4 / 25.2
//   IQ4_XS          512 15.3 / 11.0  4,096 16.7 / 11.1  6,144 16.4 / 12.3  12,288 18.2 / 18.2
// (Q6_K gained 8% at most, 12.1 / 11.1 at 2,048, and is not split.)
constexpr int64_t kSpreadQ3 = 2048, kSpreadIq4 = 6144;

template <int SRC, bool IMAT, int SQ>
hipError_t launch_iq4(const qs::KArgs& a, hipStream_t st) {
    const dim3 wave(64);
    if (a.n_units <= kSpreadIq4) return launch(qs::k_iq4_xs<SRC, IMAT, SQ, 4>, sb_grid(a, 32), wave, st, a);
    return launch(qs::k_iq4_xs<SRC, IMAT, SQ, 1>, sb_grid(a, 8), wave, st, a);
}

// SQ: the host whose square-root rounding the weights take (qs::SQ_*);
// kernels whose weights take no square root are instantiated once (SQ_IEEE).
template <int SRC, int SQ>
hipError_t launch_type(int type, bool imat, const qs::KArgs& a, hipStream_t st,
                       const IqTabs& tabs) {
    using namespace qs;
    const dim3 wave(64);
    const dim3 sb8((unsigned)((a.n_units + 7) / 8)), sb4((unsigned)((a.n_units + 3) / 4));
    switch (type) {
    case QS_TYPE_Q4_0: return launch_b32<SRC, B32::Q4_0>(a, st);
    case QS_TYPE_Q4_1: return launch_b32<SRC, B32::Q4_1>(a, st);
    case QS_TYPE_Q5_0: return launch_b32<SRC, B32::Q5_0>(a, st);
    case QS_TYPE_Q5_1: return launch_b32<SRC, B32::Q5_1>(a, st);
    case QS_TYPE_Q8_0: return launch_b32<SRC, B32::Q8_0>(a, st);
    case QS_TYPE_IQ4_NL: {
        const dim3 g((unsigned)((a.n_units + 63) / 64));
        return imat ? launch(k_iq4_nl<SRC, true, SQ>, g, wave, st, a)
                    : launch(k_iq4_nl<SRC, false, SQ_IEEE>, g, wave, st, a);
    }
    case QS_TYPE_Q4_K:
        return imat ? launch_q45<SRC, true, 15, SQ>(a, st, qkx_steps(-0.9f, 0.05f, 36, 15))
                    : launch_q45<SRC, false, 15, SQ>(a, st, qkx_steps(-1.0f, 0.1f, 20, 15));
    case QS_TYPE_Q5_K:
        return imat ? launch_q45<SRC, true, 31, SQ>(a, st, qkx_steps(-0.9f, 0.05f, 36, 31))
                    : launch_q45<SRC, false, 31, SQ>(a, st, qkx_steps(-0.5f, 0.1f, 15, 31));
    case QS_TYPE_Q6_K:
        return imat ? launch(k_q6_k<SRC, true>, sb4, wave, st, a, qx_steps(32))
                    : launch(k_q6_k<SRC, false>, sb4, wave, st, a, qx_steps(32));
    case QS_TYPE_Q3_K:
        if (!imat) return launch(k_q3_k<SRC, false, SQ_IEEE, 1>, sb4, wave, st, a, qx_steps(4), qx_steps(32));
        if (a.n_units <= kSpreadQ3)
            return launch(k_q3_k<SRC, true, SQ, 4>, sb_grid(a, 64), wave, st, a, qx_steps(4), qx_steps(32));
        return launch(k_q3_k<SRC, true, SQ, 1>, sb4, wave, st, a, qx_steps(4), qx_steps(32));
    case QS_TYPE_Q2_K:
        return imat ? launch_q2<SRC, true, SQ>(a, st, qkx_steps(-0.9f, 0.05f, 36, 3))
                    : launch_q2<SRC, false, SQ_IEEE>(a, st, qkx_steps(-0.5f, 0.1f, 15, 3));
    case QS_TYPE_IQ4_XS:
        return imat ? launch_iq4<SRC, true, SQ>(a, st) : launch_iq4<SRC, false, SQ_IEEE>(a, st);
    case QS_TYPE_IQ2_XXS: {
        // candidate numerators computed in f64 and rounded once (iq2.py:387, :470)
        QpSteps qp4{};
        IqSteps sweep{};
        int n = 0;
        for (int i = -4; i <= 4; i++)
            if (i) qp4.v[n++] = (float)(0.1 * i + 4.0);
        for (int i = -6; i <= 6; i++) sweep.v[sweep.n++] = (float)(5.0 + 0.1 * i);
        return launch(k_iq2_xxs<SRC, SQ>, sb8, wave, st, a, tabs[IQT_G2_256], qp4, sweep);
    }
    case QS_TYPE_IQ2_XS:      // SWEEP_CS iq2xs_common.py:21
        return launch(k_iq2_xs_s<SRC, false, SQ, 1>, sb4, wave, st, a, tabs[IQT_G2_512],
                      iq_steps(5.0f, 0.1f, -9, 9));
    case QS_TYPE_IQ2_S: {     // four waves per workgroup share the 1024-entry grid
        constexpr int WPG = 4;
        const dim3 g((unsigned)((a.n_units + 4 * WPG - 1) / (4 * WPG)));
        return launch(k_iq2_xs_s<SRC, true, SQ, WPG>, g, dim3(64 * WPG), st, a, tabs[IQT_G2_1024],
                      iq_steps(5.0f, 0.1f, -9, 9));
    }
    case QS_TYPE_IQ3_XXS: {    // _STEPS iq3_xxs.py:22
        const dim3 sb2((unsigned)((a.n_units + 1) / 2));
        return imat ? launch(k_iq3<SRC, false, true, SQ, 4>, sb2, wave, st, a, tabs[IQT_G3_256],
                             iq_steps(15.0f, 0.2f, -15, 15))
                    : launch(k_iq3<SRC, false, false, SQ, 4>, sb2, wave, st, a, tabs[IQT_G3_256],
                             iq_steps(15.0f, 0.2f, -15, 15));
    }
    case QS_TYPE_IQ3_S: {      // _STEPS iq3_s.py:22
        const dim3 sb2((unsigned)((a.n_units + 1) / 2));
        return imat ? launch(k_iq3<SRC, true, true, SQ, 4>, sb2, wave, st, a, tabs[IQT_G3_512],
                             iq_steps(15.0f, 0.2f, -9, 9))
                    : launch(k_iq3<SRC, true, false, SQ, 4>, sb2, wave, st, a, tabs[IQT_G3_512],
                             iq_steps(15.0f, 0.2f, -9, 9));
    }
    default:
        return hipErrorInvalidValue;
    }
}

}  // namespace

template <int SRC>
hipError_t launch_src(int sq, int type, bool imat, const qs::KArgs& a, hipStream_t st, const IqTabs& tabs) {
    switch (sq) {
    case qs::SQ_INTEL: return launch_type<SRC, qs::SQ_INTEL>(type, imat, a, st, tabs);
    case qs::SQ_AMD: return launch_type<SRC, qs::SQ_AMD>(type, imat, a, st, tabs);
    default: return launch_type<SRC, qs::SQ_IEEE>(type, imat, a, st, tabs);
    }
}


template hipError_t launch_src<QS_LAUNCH_SRC>(int, int, bool, const qs::KArgs&, hipStream_t, const IqTabs&);

}  // namespace qs_launch
