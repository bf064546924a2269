// Which tile a product of the SwiGLU block is cut into, and whether k is split over workgroups.  Host code.
#pragma once
#include <stdint.h>

#include <initializer_list>

namespace mg {

// Time of a launch = 3 us + rounds of one tile per compute unit * (cost of a tile + 64s of k * time of each), fitted to
// products with 32 to 5500 tiles of each kind (bf16, us, from the largest tile to the smallest): 7168 x 2048
// outputs, k 1024: 30 / 36 / 45 / 57; 1024 x 7168, k 2048: 46 / 32 / 34.6 / 50; 1024 x 3584, k 2048: 44 / 27 / 19.1 / 26.5;
// 1024 x 2048, k 3584: 69 / 40 / 24.5 / 21; 4096 x 11008, k 128: 28.6 / 41 / 49 / 93.
struct MlpShape { int bm, bn, bk; float tile_us, k64_us; };
constexpr MlpShape kMlpShapes[] = {{256, 256, 64, 9.0f, 1.1f}, {128, 256, 64, 4.7f, 0.68f}, {128, 128, 64, 3.7f, 0.36f}, {128, 64, 128, 2.2f, 0.31f}};

struct MlpPlan { int shape, splits; };

// A product [M, N] over K; `ragged`: K need not be a multiple of the step (lines beyond the last read as zero); `splittable`:
// the sums may be finished by a second launch, from an array of fp32 per split.  Few tokens through wide weights leave most
// compute units without a tile otherwise: 128 tokens, 4096 x 11008, forward + backward 262 us with splits, 566 without.
inline MlpPlan mlp_plan(int64_t M, int64_t N, int64_t K, bool ragged, bool splittable, int cus) {
    MlpPlan best = {-1, 1};
    float least = 0.0f;
    for (int i = 0; i < 4; ++i) {
        const MlpShape& s = kMlpShapes[i];
        if (!ragged && K % s.bk != 0) continue;
        const int64_t tiles = ((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
        for (const int splits : {1, 2, 3, 4, 6, 8}) {
            const int64_t k = (K + splits - 1) / splits;
            if (splits > 1 && (!splittable || k < 512 || splits * M * N * 4 > (256LL << 20))) break;
            float t = (float)((tiles * splits + cus - 1) / cus) * (s.tile_us + s.k64_us * (float)k / 64.0f);
            if (splits > 1) t += 8.0f + (float)(splits * M * N) * (8.0f / 5e6f);   // written and read at 5 TB/s, the launch, and stores that do not overlap
            if (best.shape < 0 || t < least) { best = {i, splits}; least = t; }
        }
    }
    return best;
}

}  // namespace mg
