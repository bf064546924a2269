// Which tile a product of the SwiGLU block is cut into, and whether k is split over workgroups.  Host code without a
// HIP header: the test of which plans there are compiles it alone.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <initializer_list>

namespace mg {

// Time of a launch = rounds of one tile per compute unit * (cost of a tile + 64s of k * time of each), in blocks whose operands
// come from memory.  Single products on cached operands (bf16, us, from the largest tile to the smallest): 7168 x 2048
// outputs, k 1024: 30 / 36 / 45 / 57; 1024 x 7168, k 2048: 46 / 32 / 34.6 / 50; 1024 x 3584, k 2048: 44 / 27 / 19.1 / 26.5;
// 1024 x 2048, k 3584: 69 / 40 / 24.5 / 21; 4096 x 11008, k 128: 28.6 / 41 / 49 / 93.  The times fitted to those (1.1, 0.68, 0.36, 0.31)
// give the medium tile too much in a block: forward + backward of 128 and 320 tokens, 4096 x 11008, 297 and 458 us
// with them, 265 and 418 with these; 742, 1664 x 4608 151.5 / 144; 1024, 2048 x 3584 159.6 / 157.3.
struct MlpShape { int bm, bn, bk; float tile_us, k64_us; };
constexpr MlpShape kMlpShapes[] = {{256, 256, 64, 9.0f, 1.3f}, {128, 256, 64, 4.7f, 0.80f}, {128, 128, 64, 3.7f, 0.47f}, {128, 64, 128, 2.2f, 0.34f}};

struct MlpPlan { int shape, splits; };

// What is known of a product [M, N] over K: `ragged`, K need not be a multiple of the step (lines beyond the last read as zero);
// `splittable`, the sums may be finished by a second launch, from an array of fp32 per split.  Few tokens through wide weights
// leave most compute units without a tile otherwise: 128 tokens, 4096 x 11008, forward + backward 262 us with splits, 566 without.
struct MlpSize { int64_t M, N, K; bool ragged, splittable; };

// One way to do it: tiles (of all splits), time of one, and what the second launch adds.
struct MlpWay { MlpPlan plan; int64_t tiles; float tile_us, extra_us; };

inline float mlp_tile_us(MlpPlan p, int64_t K) {
    const MlpShape& s = kMlpShapes[p.shape];
    return s.tile_us + s.k64_us * (float)((K + p.splits - 1) / p.splits) / 64.0f;
}

// Whether shape `i` can do it, and how if its k goes to `splits`.
inline bool mlp_way(const MlpSize& p, int i, int splits, MlpWay* way) {
    const MlpShape& s = kMlpShapes[i];
    if (!p.ragged && p.K % s.bk != 0) return false;
    if (splits > 1 && (!p.splittable || p.K / splits < 512 || splits * p.M * p.N * 4 > (256LL << 20))) return false;
    way->plan = {i, splits};
    way->tiles = ((p.M + s.bm - 1) / s.bm) * ((p.N + s.bn - 1) / s.bn) * splits;
    way->tile_us = mlp_tile_us(way->plan, p.K);
    // written and read at 5 TB/s, the launch, and stores that do not overlap
    way->extra_us = splits > 1 ? 6.0f + (float)(splits * p.M * p.N) * (8.0f / 5e6f) : 0.0f;
    return true;
}
constexpr int kMlpSplits[] = {1, 2, 3, 4, 6, 8};

inline MlpPlan mlp_plan(const MlpSize& p, int cus, float* us = nullptr) {
    MlpPlan best = {-1, 1};
    float least = 0.0f;
    for (int i = 0; i < 4; ++i)
        for (const int splits : kMlpSplits) {
            MlpWay w;
            if (!mlp_way(p, i, splits, &w)) break;
            const float t = (float)((w.tiles + cus - 1) / cus) * w.tile_us + w.extra_us;
            if (best.shape < 0 || t < least) { best = w.plan; least = t; }
        }
    if (us != nullptr) *us = least;
    return best;
}

// When the last of `a`'s tiles and then `b`'s, each taking the first compute unit that is free, is done.
inline float mlp_makespan(const MlpWay& a, const MlpWay& b, int cus) {
    const int64_t full = a.tiles / cus, more = a.tiles % cus;      // `more` units are free a tile later than the others
    const float early = (float)full * a.tile_us, late = early + a.tile_us;
    float low = more > 0 ? late : early, high = late + (float)((b.tiles + cus - 1) / cus) * b.tile_us;
    for (int i = 0; i < 8 && high - low > 0.5f; ++i) {
        const float t = 0.5f * (low + high);
        const int64_t done = more * (t > late ? (int64_t)((t - late) / b.tile_us) : 0) + (cus - more) * (int64_t)((t - early) / b.tile_us);
        if (done >= b.tiles) high = t;
        else low = t;
    }
    return high;
}

// The plans of two products that share a launch, longer tiles first: for the pair a cheaper tile often beats the one that fills
// the compute units by itself.
inline void mlp_plan_pair(const MlpSize& p, const MlpSize& q, int cus, MlpPlan* plan_p, MlpPlan* plan_q) {
    float least = -1.0f;
    MlpWay ways[2][24];
    int count[2] = {0, 0};
    const MlpSize* sizes[2] = {&p, &q};
    for (int k = 0; k < 2; ++k)
        for (int i = 0; i < 4; ++i)
            for (const int splits : kMlpSplits) {
                MlpWay w;
                if (!mlp_way(*sizes[k], i, splits, &w)) break;
                // of the split ways only those that still leave units free without
                if (splits > 1 && w.tiles / splits * (splits - 1) > 2 * cus) break;
                ways[k][count[k]++] = w;
            }
    for (int i = 0; i < count[0]; ++i)
        for (int k = 0; k < count[1]; ++k) {
            const MlpWay &a = ways[0][i], &b = ways[1][k];
            const float work = ((float)a.tiles * a.tile_us + (float)b.tiles * b.tile_us) / (float)cus + a.extra_us + b.extra_us;
            if (least >= 0.0f && work >= least) continue;      // no order can be better
            const float t = (a.tile_us >= b.tile_us ? mlp_makespan(a, b, cus) : mlp_makespan(b, a, cus)) + a.extra_us + b.extra_us;
            if (least < 0.0f || t < least) { least = t; *plan_p = a.plan; *plan_q = b.plan; }
        }
}

// The block's products: [gate | up] with the activation, the second projection; the activation's gradient, that of an input, that of
// weights.
enum class MlpWhat { gate_up, down, activation_bwd, input_grad, weight_grad };
inline MlpSize mlp_size(MlpWhat what, int64_t M, int64_t N, int64_t K) {
    const bool fused = what == MlpWhat::gate_up || what == MlpWhat::activation_bwd;   // the activation needs whole sums
    return {M, what == MlpWhat::gate_up ? 2 * N : N, K, what == MlpWhat::weight_grad, !fused};
}
inline int64_t mlp_partial_bytes(MlpPlan p, int64_t M, int64_t N) { return p.splits > 1 ? p.splits * M * N * 4 : 0; }

struct MlpForward {
    float us[2];           // expected
    MlpPlan gate_up, down;
    int64_t workspace;
    MlpForward(int64_t t, int64_t d, int64_t h, int cus)
        : gate_up(mlp_plan(mlp_size(MlpWhat::gate_up, t, h, d), cus, &us[0])), down(mlp_plan(mlp_size(MlpWhat::down, t, d, h), cus, &us[1])),
          workspace(mlp_partial_bytes(down, t, d)) {}
};

// Whether the two launches of a forward pass that no backward pass follows take no more time than the library's products
// and the activation, on the 256 compute units that both sides were measured on (700 sizes: 20 to 65536 tokens, 3 to 425 MB of
// weights, replayed graphs, bf16 and fp16).  The library's time scatters by 10 % around the line below, which lies where least
// is lost on either side; up to the given weights these products win or are level at every number of tokens measured:
//   below 24 MB: 512 x 1024 17.2 / 14.6 us at 65 tokens, 285 / 230 at 65536; 1024 x 2816 19.0 / 18.6, 1042 / 977;
//   below 60 MB and 5000 tokens: 2048 x 3584 1024 tokens 64.9 / 54.4, 4096 168 / 160, but 8192 297 / 302; 1664 x 4608 1800 tokens 124 / 107;
//   beyond: 4096 x 11008 256 tokens 118 / 109, but 320 134 / 146 and 384 145 / 158 (row tiles that just miss), 448 168 / 157; 4096 x 6912 256
//     87 / 76, 640 131 / 146, 768 141 / 162, 2048 293 / 298; 4096 x 5440 65536 tokens 6090 / 6531; 8192 x 2048 64 tokens 41 / 56.
// Of the sizes taken 1 in 100 is more than 2 % slower (worst 256 tokens, 8192 x 2048, 63 / 66).  Between 20 and 130 tokens sizes of less
// than 40 us, where three operators take 47 us on the host, are taken although a replayed graph may lose 1 to 6 us (65 tokens, 1536 x 2560
// 18.6 / 22.6, eager 46 / 20).  Wins given up: 5 to 20 % at some sizes beyond 60 MB and 640 tokens (2048, 4096 x 11008 588 / 462).
inline bool mlp_forward_wins(int64_t t, int64_t d, int64_t h) {
    const float mb = 6e-6f * (float)d * (float)h;
    if (mb <= 24.0f || (mb <= 60.0f && t <= 5000)) return true;
    const MlpForward pass(t, d, h, 256);
    const float library_us = 20.0f + 30.0f * (float)std::min<int64_t>(t, 256) / 256.0f + 0.15f * mb + mb * (float)t / 2000.0f;
    return pass.us[0] + pass.us[1] <= library_us;
}

// Two launches: the gradients of w3 and, through the activation, of [gate | up]; then those of w12 and x.
struct MlpBackward {
    MlpPlan w3{-1, 1}, act{-1, 1}, w12{-1, 1}, x{-1, 1};
    int64_t workspace[2], at[2];   // bytes of each launch, and where its second product's begin
    MlpBackward(int64_t t, int64_t d, int64_t h, bool want_x, bool want_12, bool want_3, int cus) {
        const MlpSize s3 = mlp_size(MlpWhat::weight_grad, d, h, t), sa = mlp_size(MlpWhat::activation_bwd, t, h, d);
        const MlpSize s12 = mlp_size(MlpWhat::weight_grad, 2 * h, d, t), sx = mlp_size(MlpWhat::input_grad, t, d, 2 * h);
        const bool want_a = want_x || want_12;
        if (want_3 && want_a) mlp_plan_pair(s3, sa, cus, &w3, &act);
        else if (want_3) w3 = mlp_plan(s3, cus);
        else if (want_a) act = mlp_plan(sa, cus);
        if (want_12 && want_x) mlp_plan_pair(s12, sx, cus, &w12, &x);
        else if (want_12) w12 = mlp_plan(s12, cus);
        else if (want_x) x = mlp_plan(sx, cus);
        at[0] = mlp_partial_bytes(w3, d, h);
        workspace[0] = at[0];
        at[1] = mlp_partial_bytes(w12, 2 * h, d);
        workspace[1] = at[1] + mlp_partial_bytes(x, t, d);
    }
    int64_t needs() const { return std::max(workspace[0], workspace[1]); }
};

}  // namespace mg
