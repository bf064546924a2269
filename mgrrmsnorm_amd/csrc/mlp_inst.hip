// Launchers of the SwiGLU block's products (fp16 and bf16): MG_DTYPE picks the type.
#include "megagemm_hip.h"
#include "mg_launch.hpp"
#include "mlp_gemm.hpp"

namespace mg {
namespace {

#if MG_DTYPE == 1
using T = half_t;
#else
using T = bf16_t;
#endif

// Four tiles, from the most reuse of what LDS holds to the most workgroups.  Eight waves each, so that two share a SIMD
// and one's LDS reads go beside the other's matrix instructions; 128 KiB of LDS and more, one workgroup per compute unit.
using Huge = MlpCfg<256, 256, 64, 2, 4, 1, 2>;
using Large = MlpCfg<128, 256, 64, 2, 4, 1, 3>;
using Medium = MlpCfg<128, 128, 64, 2, 2, 2, 4>;
using Small = MlpCfg<128, 64, 128, 2, 1, 4, 3>;

template <int I, class C> constexpr bool is_shape() {
    return kMlpShapes[I].bm == C::BM && kMlpShapes[I].bn == C::BN && kMlpShapes[I].bk == C::BK;
}
static_assert(is_shape<0, Huge>() && is_shape<1, Large>() && is_shape<2, Medium>() && is_shape<3, Small>(), "the plan's tiles");

template <class C, bool A_ALONG_K, bool B_ALONG_K, int WHAT>
hipError_t run(const MlpArgs& a, int splits, hipStream_t s) {
    constexpr int BN = WHAT == kMlpGateUp ? C::BN / 2 : C::BN;
    const unsigned rows = (a.M + C::BM - 1) / C::BM, cols = (a.N + BN - 1) / BN;
    const MlpOperand A = {a.a, a.a_bytes, a.a_ld}, B = {a.b, a.b_bytes, a.b_ld};
    const MlpOut o = {WHAT == kMlpPartial ? a.partial : a.out, a.second, a.in, a.M, a.N};
    return launch(mlp_gemm<T, C, A_ALONG_K, B_ALONG_K, WHAT>, dim3(rows * cols * splits), dim3(C::THREADS), 0, s, A, B, o, a.K, splits);
}

template <bool A_ALONG_K, bool B_ALONG_K, int WHAT>
hipError_t by_shape(const MlpArgs& a, MlpPlan p, hipStream_t s) {
    switch (p.shape) {
        case 0: return run<Huge, A_ALONG_K, B_ALONG_K, WHAT>(a, p.splits, s);
        case 1: return run<Large, A_ALONG_K, B_ALONG_K, WHAT>(a, p.splits, s);
        case 2: return run<Medium, A_ALONG_K, B_ALONG_K, WHAT>(a, p.splits, s);
        case 3: return run<Small, A_ALONG_K, B_ALONG_K, WHAT>(a, p.splits, s);
        default: return hipErrorInvalidValue;
    }
}

template <bool A_ALONG_K, bool B_ALONG_K>
hipError_t maybe_split(const MlpArgs& a, MlpPlan p, hipStream_t s) {
    if (p.splits == 1) return by_shape<A_ALONG_K, B_ALONG_K, kMlpStore>(a, p, s);
    const hipError_t e = by_shape<A_ALONG_K, B_ALONG_K, kMlpPartial>(a, p, s);
    if (e != hipSuccess) return e;
    const unsigned vectors = (unsigned)((long)a.M * a.N / 8);
    return launch(mlp_add<T>, dim3((vectors + 255) / 256), dim3(256), 0, s, (T*)a.out, (const float*)a.partial, vectors, p.splits);
}

}  // namespace

template <>
hipError_t launch_mlp<T>(MlpWhat what, const MlpArgs& a, MlpPlan p, hipStream_t s) {
    switch (what) {
        case MlpWhat::gate_up: return by_shape<true, true, kMlpGateUp>(a, p, s);
        case MlpWhat::down: return maybe_split<true, true>(a, p, s);
        case MlpWhat::activation_bwd: return by_shape<true, false, kMlpActBwd>(a, p, s);
        case MlpWhat::input_grad: return maybe_split<true, false>(a, p, s);
        case MlpWhat::weight_grad: return maybe_split<false, false>(a, p, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace mg
