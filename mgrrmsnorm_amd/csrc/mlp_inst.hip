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
using Large = MlpCfg<256, 128, 64, 4, 2, 1, 3>;
using Medium = MlpCfg<128, 128, 64, 2, 4, 1, 4>;
using Small = MlpCfg<128, 64, 128, 2, 2, 2, 3>;

// Time of a launch = rounds of one tile per compute unit * (cost of a tile + 64s of k * time of each), fitted to
// 15 and 30 GFLOP products with 32 to 896 tiles of each kind (bf16, us): 7168 x 2048 outputs, k 1024: 29.4 / 34.5 / 40 / 53 from
// the largest tile to the smallest; 1024 x 7168, k 2048: 42.6 / 29.8 / 34.6 / 45.9; 1024 x 3584, k 2048: 42.7 / 26.3 / 19.8 / 25.6;
// 1024 x 2048, k 3584: 69 / 39.8 / 25.9 / 20.1.
struct Shape { int bm, bn, bk; float tile_us, k64_us; };
constexpr Shape kShapes[] = {{Huge::BM, Huge::BN, Huge::BK, 7.0f, 1.15f},
                             {Large::BM, Large::BN, Large::BK, 4.7f, 0.68f},
                             {Medium::BM, Medium::BN, Medium::BK, 4.0f, 0.37f},
                             {Small::BM, Small::BN, Small::BK, 0.5f, 0.33f}};

// `k_ragged`: k need not be a multiple of the step (lines beyond the last read as zero)
int pick(const MlpArgs& a, int columns, bool k_ragged) {
    int best = -1;
    float least = 0.0f;
    for (int i = 0; i < 4; ++i) {
        const Shape& s = kShapes[i];
        if (!k_ragged && a.K % s.bk != 0) continue;
        const long tiles = (long)((a.M + s.bm - 1) / s.bm) * ((columns + s.bn - 1) / s.bn);
        const float t = (float)((tiles + a.cus - 1) / a.cus) * (s.tile_us + s.k64_us * (float)a.K / 64.0f);
        if (best < 0 || t < least) { best = i; least = t; }
    }
    return best;
}

template <class C, bool A_ALONG_K, bool B_ALONG_K, int WHAT>
hipError_t run(const MlpArgs& a, hipStream_t s) {
    constexpr int BN = WHAT == kMlpGateUp ? C::BN / 2 : C::BN;
    const unsigned rows = (a.M + C::BM - 1) / C::BM, cols = (a.N + BN - 1) / BN;
    const MlpOperand A = {a.a, a.a_bytes, a.a_ld}, B = {a.b, a.b_bytes, a.b_ld};
    const MlpOut o = {a.out, a.second, a.in, a.M, a.N};
    return launch(mlp_gemm<T, C, A_ALONG_K, B_ALONG_K, WHAT>, dim3(rows * cols), dim3(C::THREADS), 0, s, A, B, o, a.K, 8);
}

template <bool A_ALONG_K, bool B_ALONG_K, int WHAT>
hipError_t by_shape(const MlpArgs& a, hipStream_t s) {
    switch (pick(a, WHAT == kMlpGateUp ? 2 * a.N : a.N, !A_ALONG_K && !B_ALONG_K)) {
        case 0: return run<Huge, A_ALONG_K, B_ALONG_K, WHAT>(a, s);
        case 1: return run<Large, A_ALONG_K, B_ALONG_K, WHAT>(a, s);
        case 2: return run<Medium, A_ALONG_K, B_ALONG_K, WHAT>(a, s);
        case 3: return run<Small, A_ALONG_K, B_ALONG_K, WHAT>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

template <>
hipError_t launch_mlp<T>(MlpWhat what, const MlpArgs& a, hipStream_t s) {
    switch (what) {
        case MlpWhat::gate_up: return by_shape<true, true, kMlpGateUp>(a, s);
        case MlpWhat::down: return by_shape<true, true, kMlpStore>(a, s);
        case MlpWhat::activation_bwd: return by_shape<true, false, kMlpActBwd>(a, s);
        case MlpWhat::input_grad: return by_shape<true, false, kMlpStore>(a, s);
        case MlpWhat::weight_grad: return by_shape<false, false, kMlpStore>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace mg
