// Launchers of the SwiGLU block's projections (fp16 and bf16).
#include "megagemm_hip.h"
#include "mg_launch.hpp"
#include "skinny_gemm.hpp"

namespace mg {
namespace {

template <typename T, int MB, int NT, int WAVES, int U, bool PAIRED>
hipError_t run(const SkinnyArgs& a, hipStream_t s) {
    const unsigned grid = (unsigned)(a.N < a.cus ? a.N : a.cus);
    return launch(skinny_gemm<T, MB, NT, WAVES, U, PAIRED>, dim3(grid), dim3(WAVES * kWave), 0, s, (T*)a.out, (const T*)a.x,
                  (const T*)a.w, a.tokens, a.K, a.N);
}

// The tiles of 16 weight rows that a workgroup's share of the columns needs decide how many of
// them go together: with one or two there are registers for 16 waves, with more the tiles keep
// enough bytes in flight on 8 (hidden = 3072, d_model = 1152, 8 tokens, two tiles: 5.6 us with
// MB = 2 on 16 waves, 6.1 with MB = 4 on 8; second projection at d_model = 4096, one tile: 13.0 with
// MB = 1 on 16 waves, 14.9 with MB = 4 on 8).  Beyond 16 tokens the activations take the registers of
// the other 8 waves.
template <typename T, int NT, bool PAIRED>
hipError_t by_share(const SkinnyArgs& a, hipStream_t s) {
    const int share = (a.N + a.cus - 1) / a.cus;
    const int tiles = (share + (PAIRED ? 7 : 15)) / (PAIRED ? 8 : 16);
    constexpr int WAVES = NT == 1 ? 16 : 8;
    if (tiles <= 1) return run<T, 1, NT, WAVES, NT == 1 ? 2 : 4, PAIRED>(a, s);
    if (tiles == 2) return run<T, 2, NT, WAVES, 2, PAIRED>(a, s);
    return run<T, 4, NT, 8, NT == 4 ? 1 : 2, PAIRED>(a, s);   // four by four tiles with two steps: spills
}

template <typename T, bool PAIRED>
hipError_t by_tokens(const SkinnyArgs& a, hipStream_t s) {
    if (a.tokens <= 16) return by_share<T, 1, PAIRED>(a, s);
    if (a.tokens <= 32) return by_share<T, 2, PAIRED>(a, s);
    if (a.tokens <= 48) return by_share<T, 3, PAIRED>(a, s);
    return by_share<T, 4, PAIRED>(a, s);
}

}  // namespace

hipError_t launch_skinny_gemm(int dtype, bool paired, const SkinnyArgs& a, hipStream_t s) {
    if (a.tokens < 1 || a.tokens > kSkinnyMaxTokens || a.K < 8 || a.K % 8 != 0 || a.N < 1 || a.cus < 1) return hipErrorInvalidValue;
    switch (dtype) {
        case MG_F16: return paired ? by_tokens<half_t, true>(a, s) : by_tokens<half_t, false>(a, s);
        case MG_BF16: return paired ? by_tokens<bf16_t, true>(a, s) : by_tokens<bf16_t, false>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mg
