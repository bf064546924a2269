// Launchers of the SwiGLU block's projections (fp16 and bf16).
#include "megagemm_hip.h"
#include "mg_launch.hpp"
#include "skinny_gemm.hpp"

namespace mg {
namespace {

template <typename T, int MB, int WAVES, int U, bool PAIRED>
hipError_t run(const SkinnyArgs& a, hipStream_t s) {
    const unsigned grid = (unsigned)(a.N < a.cus ? a.N : a.cus);
    return launch(skinny_gemm<T, MB, WAVES, U, PAIRED>, dim3(grid), dim3(WAVES * kWave), 0, s, (T*)a.out, (const T*)a.x,
                  (const T*)a.w, a.tokens, a.K, a.N);
}

// The tiles of 16 weight rows that a workgroup's share of the columns needs decide how many of
// them go together: with one or two there are registers for 16 waves, with more the tiles keep
// enough bytes in flight on 8 (hidden = 3072, d_model = 1152, 8 tokens, two tiles: 5.6 us with
// MB = 2 on 16 waves, 6.1 with MB = 4 on 8; second projection at d_model = 4096, one tile: 13.0 with
// MB = 1 on 16 waves, 14.9 with MB = 4 on 8).
template <typename T, bool PAIRED>
hipError_t by_share(const SkinnyArgs& a, hipStream_t s) {
    const int share = (a.N + a.cus - 1) / a.cus;
    const int tiles = (share + (PAIRED ? 7 : 15)) / (PAIRED ? 8 : 16);
    if (tiles <= 1) return run<T, 1, 16, 2, PAIRED>(a, s);
    if (tiles == 2) return run<T, 2, 16, 2, PAIRED>(a, s);
    return run<T, 4, 8, 2, PAIRED>(a, s);
}

}  // namespace

hipError_t launch_skinny_gemm(int dtype, bool paired, const SkinnyArgs& a, hipStream_t s) {
    if (a.tokens < 1 || a.tokens > kSkinnyMaxTokens || a.K < 8 || a.K % 8 != 0 || a.N < 1 || a.cus < 1) return hipErrorInvalidValue;
    switch (dtype) {
        case MG_F16: return paired ? by_share<half_t, true>(a, s) : by_share<half_t, false>(a, s);
        case MG_BF16: return paired ? by_share<bf16_t, true>(a, s) : by_share<bf16_t, false>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mg
