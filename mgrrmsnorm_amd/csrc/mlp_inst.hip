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

template <int SHAPE> struct ShapeOf;
template <> struct ShapeOf<0> { using type = Huge; };
template <> struct ShapeOf<1> { using type = Large; };
template <> struct ShapeOf<2> { using type = Medium; };
template <> struct ShapeOf<3> { using type = Small; };

MlpJob job_of(const MlpArgs& a, MlpPlan p, bool paired) {
    const MlpShape& s = kMlpShapes[p.shape];
    const int bn = paired ? s.bn / 2 : s.bn;
    const u32 tiles = (u32)((a.M + s.bm - 1) / s.bm) * (u32)((a.N + bn - 1) / bn) * (u32)p.splits;
    return {{a.a, a.a_bytes, a.a_ld}, {a.b, a.b_bytes, a.b_ld}, {p.splits > 1 ? a.partial : a.out, a.second, a.in, a.M, a.N}, a.K, p.splits, p.shape, tiles};
}

// ---- forward: one product a launch, each the other's input ----
template <int SHAPE, int WHAT>
hipError_t run(const MlpJob& job, const MlpWarm& warm, u32 idle, hipStream_t s) {
    using C = typename ShapeOf<SHAPE>::type;
    return launch(mlp_gemm<T, C, true, true, WHAT>, dim3(job.tiles + idle), dim3(C::THREADS), 0, s, job, warm);
}
template <int WHAT>
hipError_t by_shape(const MlpJob& job, hipStream_t s, const MlpWarm& warm = {}, u32 idle = 0) {
    switch (job.shape) {
        case 0: return run<0, WHAT>(job, warm, idle, s);
        case 1: return run<1, WHAT>(job, warm, idle, s);
        case 2: return run<2, WHAT>(job, warm, idle, s);
        case 3: return run<3, WHAT>(job, warm, idle, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t add_parts(const MlpArgs& a, MlpPlan p, hipStream_t s) {
    if (p.splits == 1) return hipSuccess;
    const unsigned vectors = (unsigned)((long)a.M * a.N / 8);
    return launch(mlp_add<T>, dim3((vectors + 255) / 256), dim3(256), 0, s, (T*)a.out, (const float*)a.partial, vectors, p.splits);
}

// ---- backward: two products a launch ----
// Neither needs the other, and each alone leaves compute units idle: at 1024 tokens, 2048 x 3584, 224 tiles for 256 of them and a
// ramp, a tail and a launch of its own.  There the four launches took 22.4 + 21 and 39.3 + 33.9 us, the two take 36 and
// 65, and a whole step 156.3 us instead of 168.6; 300 tokens, 512 x 1024 37.8 instead of 47 (eager: launches).  Longer tiles
// first, whichever product they are of.  Every kind and size of tile is in the one kernel, which all of them suit: 512
// threads, one workgroup per compute unit.
enum Kind { kWeightGrad, kInputGrad, kActBwd };
constexpr int kBackwardLds = 3 * 48 * 1024;
static_assert(Huge::STAGE * Huge::STAGES <= kBackwardLds && Large::STAGE * Large::STAGES <= kBackwardLds && Medium::STAGE * Medium::STAGES <= kBackwardLds &&
              Small::STAGE * Small::STAGES <= kBackwardLds && Huge::THREADS == 512 && Large::THREADS == 512 && Medium::THREADS == 512 && Small::THREADS == 512, "");

template <class C>
__device__ __forceinline__ void any_kind(const MlpJob& job, int kind, u32 id, char MG_LDS* lds) {
    if (kind == kWeightGrad) {
        if (job.splits > 1) mlp_job<T, C, false, false, kMlpPartial>(job, id, lds);
        else mlp_job<T, C, false, false, kMlpStore>(job, id, lds);
    } else if (kind == kInputGrad) {
        if (job.splits > 1) mlp_job<T, C, true, false, kMlpPartial>(job, id, lds);
        else mlp_job<T, C, true, false, kMlpStore>(job, id, lds);
    } else {
        mlp_job<T, C, true, false, kMlpActBwd>(job, id, lds);
    }
}

// `a_blocks` workgroups for job a, a multiple of 8 so that both keep their tiles' dies
__global__ void __launch_bounds__(512, 2)
mlp_backward(MlpJob a, int a_kind, u32 a_blocks, MlpJob b, int b_kind) {
    __shared__ __attribute__((aligned(1024))) char lds[kBackwardLds];
    const bool second = blockIdx.x >= a_blocks;
    const MlpJob& job = second ? b : a;
    const int kind = second ? b_kind : a_kind;
    const u32 id = second ? blockIdx.x - a_blocks : blockIdx.x;
    if (id >= job.tiles) return;
    switch (job.shape) {
        case 0: return any_kind<Huge>(job, kind, id, (char MG_LDS*)lds);
        case 1: return any_kind<Large>(job, kind, id, (char MG_LDS*)lds);
        case 2: return any_kind<Medium>(job, kind, id, (char MG_LDS*)lds);
        case 3: return any_kind<Small>(job, kind, id, (char MG_LDS*)lds);
    }
}

Kind kind_of(MlpWhat what) {
    return what == MlpWhat::weight_grad ? kWeightGrad : what == MlpWhat::input_grad ? kInputGrad : kActBwd;
}

}  // namespace

template <>
hipError_t launch_mlp_forward<T>(MlpWhat what, const MlpArgs& a, MlpPlan p, hipStream_t s) {
    const MlpJob job = job_of(a, p, what == MlpWhat::gate_up);
    if (what == MlpWhat::gate_up) {
        // Compute units without a tile in the last round read what the next launch wants, as much as they can in a tile's time,
        // where the weights of both leave memory idle half of the time: 1024 tokens, 2048 x 3584 160.7 -> 156.9 us forward
        // + backward, 742, 1664 x 4608 145.7 / 140.1; else the tiles wait for it, 128 tokens, 4096 x 11008 266 / 277.
        const u32 cus = (u32)a.cus, spare = (cus - job.tiles % cus) % cus;
        const float us = (float)((job.tiles + cus - 1) / cus) * mlp_tile_us(p, a.K), can = (float)spare * mlp_tile_us(p, a.K) * 40e3f;
        const u32 idle = 3.0f * (float)a.next_bytes <= us * 2.5e6f ? spare : 0u;
        const MlpWarm warm = {a.next, can < (float)a.next_bytes ? (u32)can : a.next_bytes};
        return by_shape<kMlpGateUp>(job, s, warm, idle);
    }
    if (p.splits == 1) return by_shape<kMlpStore>(job, s);
    const hipError_t e = by_shape<kMlpPartial>(job, s);
    return e == hipSuccess ? add_parts(a, p, s) : e;
}

template <>
hipError_t launch_mlp_backward<T>(const MlpTask* tasks, int count, hipStream_t s) {
    if (count < 1 || count > 2) return hipErrorInvalidValue;
    MlpJob jobs[2] = {job_of(tasks[0].args, tasks[0].plan, false), {}};
    if (count == 2) jobs[1] = job_of(tasks[1].args, tasks[1].plan, false);
    const int last = count - 1;
    const int first = count == 2 && mlp_tile_us(tasks[1].plan, tasks[1].args.K) > mlp_tile_us(tasks[0].plan, tasks[0].args.K) ? 1 : 0;
    const int second = count == 2 ? 1 - first : 0;
    const u32 a_blocks = (jobs[first].tiles + 7) / 8 * 8, b_blocks = count == 2 ? jobs[second].tiles : 0;
    hipError_t e = launch(mlp_backward, dim3(a_blocks + b_blocks), dim3(512), 0, s, jobs[first], (int)kind_of(tasks[first].what), a_blocks,
                          jobs[second], (int)kind_of(tasks[second].what));
    for (int i = 0; i <= last && e == hipSuccess; ++i) e = add_parts(tasks[i].args, tasks[i].plan, s);
    return e;
}

}  // namespace mg
