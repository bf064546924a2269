// The products of the SwiGLU block on the matrix cores: out[m, n] = sum_k a[m, k] * b[n, k] with either
// operand stored with k or with its rows consecutive, and the activation or its backward folded into the
// products that produce its inputs.
#pragma once
#include "mg_device.hpp"
#include "skinny_gemm.hpp"

namespace mg {

#define MG_LDS __attribute__((address_space(3)))
typedef short s16x4 __attribute__((ext_vector_type(4)));

// A byte offset that is outside every buffer here (they are below 2 GiB).
constexpr u32 kNowhere = 0xFFFFFF00u;

// One operand in memory: `bytes` long from `p`, `ld` elements from one line to the next.
struct MlpOperand { const void* p; u32 bytes; int ld; };

// BM x BN outputs per workgroup, BK of k per step; the tile is split over WM x WN waves, and each step's k
// over WK groups of them; STAGES steps of both operands in LDS.
template <int BM_, int BN_, int BK_, int WM_, int WN_, int WK_, int STAGES_>
struct MlpCfg {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, WK = WK_, STAGES = STAGES_;
    static constexpr int WAVES = WM * WN * WK, THREADS = WAVES * kWave;
    static constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;   // a wave's tile, in fragments
    static constexpr int SUBSTEPS = BK / 32 / WK;                                  // of one matrix instruction in k
    static constexpr int A_BYTES = BM * BK * 2, STAGE = (BM + BN) * BK * 2;
    static_assert(BK / 32 % WK == 0 && (SUBSTEPS == 1 || SUBSTEPS == 2), "");
    static_assert(STAGE * STAGES <= 160 * 1024, "LDS of a compute unit");
};

// ROWS x BK elements of one operand on their way from memory to LDS, without passing through registers: each
// request puts 16 bytes per lane at consecutive LDS addresses, so the order in LDS is made by choosing what
// each lane asks for.  ALONG_K: lines of BK elements, one per row; else lines of ROWS elements, one per k.
// A line's 16-byte units (its 32-byte pairs of units) are permuted by exclusive-or with bits of the line's
// number, so that the lines a fragment is read from lie in different banks (64 of 4 bytes).
// PAIRED: half of the rows of every TN are taken from `hidden` rows further on (gate and up of the same columns).
template <int ROWS, int BK, int THREADS, bool ALONG_K, int TN = 0>
struct MlpTile {
    static constexpr int N = ROWS * BK * 2 / 16 / THREADS;   // requests per thread
    static_assert(N * 16 * THREADS == ROWS * BK * 2, "whole requests");
    static constexpr int UNITS = (ALONG_K ? BK : ROWS) / 8;  // 16-byte units in a line
    u32 off[N];

    static __device__ __forceinline__ int permute(int line) {
        if constexpr (ALONG_K) return BK == 64 ? (line >> 1) & 7 : line & 15;         // two lines / one line in 256 bytes
        else if constexpr (ROWS >= 128) return (line & 3) | ((line >> 3) & 1) << 2;   // lines 0-3, 8-11, ... read together
        else return ((line >> 1) & 1) | ((line >> 3) & 1) << 1;
    }
    __device__ __forceinline__ void init(int tid, int row0, int ld, int hidden) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int at = i * THREADS + tid;
            const int line = at / UNITS, unit = at % UNITS;
            if constexpr (ALONG_K) {
                int row = row0 + line;
                if constexpr (TN > 0) row = row0 + line / TN * (TN / 2) + line % (TN / 2) + (line % TN >= TN / 2 ? hidden : 0);
                off[i] = (u32)row * (u32)ld * 2u + (u32)((unit ^ permute(line)) * 16);
            } else {
                const int u = ((unit >> 1) ^ permute(line)) * 2 + (unit & 1);
                off[i] = (u32)line * (u32)ld * 2u + (u32)(row0 * 2 + u * 16);
            }
        }
    }
    // bytes from one step of k to the next
    static __device__ __forceinline__ u32 step(int ld) { return ALONG_K ? BK * 2u : (u32)ld * (BK * 2u); }
    __device__ __forceinline__ void request(char MG_LDS* to, rsrc_t r, int wave) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (MG_LDS void*)(to + (i * THREADS + wave * kWave) * 16), 16, (int)off[i], 0, 0, 0);
    }
    __device__ __forceinline__ void advance(u32 by) {
#pragma unroll
        for (int i = 0; i < N; ++i) off[i] += by;
    }
    // Where in the tile this lane's part of the fragment lies that covers 16 rows from `row` on and k from 32 * kk on.
    static __device__ __forceinline__ int fragment(int row, int lane, int kk) {
        if constexpr (ALONG_K) {
            const int line = row + (lane & 15);
            return line * BK * 2 + (((kk * 4 + (lane >> 4)) ^ permute(line)) << 4);
        } else {
            const int line = kk * 32 + 8 * (lane >> 4) + ((lane & 15) >> 2);
            return line * ROWS * 2 + (((row / 16) ^ permute(line)) << 5) + (lane & 3) * 8;
        }
    }
    // The same, `s` fragments of k further on: kk was a multiple of 2 (of 1 for s = 0).
    static __device__ __forceinline__ int further(int at, int s) { return ALONG_K ? at ^ (s << 6) : at + s * (32 * ROWS * 2); }
    static __device__ __forceinline__ u32x4 read(const char MG_LDS* tile, int at) {
        if constexpr (ALONG_K) {
            return *(const u32x4 MG_LDS*)(tile + at);
        } else {   // four lines of 16 elements per 16 lanes, transposed: a lane gets one column of them
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 MG_LDS*)(tile + at));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 MG_LDS*)(tile + at + 4 * ROWS * 2));
            return __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
};

// Waits until at most OUTSTANDING of this wave's requests and none of its LDS accesses are under way.
template <int OUTSTANDING>
__device__ __forceinline__ void wait_requests() {
    static_assert(OUTSTANDING < 64, "the counter's range");
    __builtin_amdgcn_s_waitcnt((OUTSTANDING & 15) | (OUTSTANDING >> 4) << 14 | 7 << 4);
}
// A barrier that accesses through these pointers do not cross.  The functions between two of them declare that theirs do not
// alias, which holds from one barrier to the next (the compiler would otherwise wait for every request before any LDS read).
__device__ __forceinline__ void step_barrier(const char MG_LDS* a, const char MG_LDS* b) {
    asm volatile("" ::"s"(a), "s"(b) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::"s"(a), "s"(b) : "memory");
}

template <class C> struct MlpFragments { u32x4 a[C::FM], b[C::FN]; };
template <class C> struct MlpSums { f32x4 v[C::FM][C::FN]; };
// What a wave has of the finished sums: a WKth of its tile's rows, the one after those of the groups before its own.
template <class C> struct MlpShare { f32x4 v[C::FM / C::WK][C::FN]; };

// One workgroup's product, bound by LDS (128 bytes a cycle).  Of the 1024 cycles that the matrix instructions of a
// 128 x 256 x 64 step take on eight waves of 64 x 64, its fragments need 1024 and its arrival from memory 384; measured 0.66 us.
// Smaller tiles can have waves as large by sharing a step's k between groups of waves: 128 x 128 on four of 64 x 64 twice over
// 18.5 us for 1024 x 3584 outputs, k 2048, against 19.8 on eight of 64 x 32 (at 128 x 256 it is no gain in a whole block,
// where the operands come from memory: 36.3 against 34.1 us for gate and up).  The loop keeps memory, LDS and matrix cores
// going at once: requests STAGES steps ahead, fragments one instruction's worth of k, and one barrier a step for both the arrival
// and the reuse of a stage.  What loses (1024 x 7168 outputs, k 2048): reads and multiplications in separate blocks 33.7
// against 31.6 us, s_setprio around the multiplications 35.1, the same tile on four waves 43 (one wave a SIMD leaves its matrix
// core waiting); on the whole block, the tiles' k started at different places 184-198 against 179 us; one 4-byte request per
// line four steps further ahead, 93 -> 100 us for 1024 x 2048, k 7168.
// At 1024 tokens, 2048 x 3584 (us, these / the library's): gate and up with the activation 34 / 35 + 4, second projection
// 26 / 25, gradient of h with the activation's 22.5 / 27 + 8, of x 39 / 52, of w3 21 / 26, of w12 34 / 42.
// `sums.v[i][j][q]` of a wave becomes out[m, n] with
//   m = m0 + wm * TM + i * 16 + lane % 16,   n = n0 + wn * TN + j * 16 + 4 * (lane / 16) + q
// (b is the instruction's first operand: a lane then owns four consecutive n and stores 8 bytes).
template <typename T, class C, bool A_ALONG_K, bool B_ALONG_K, bool PAIRED>
struct MlpProduct {
    using TA = MlpTile<C::BM, C::BK, C::THREADS, A_ALONG_K>;
    using TB = MlpTile<C::BN, C::BK, C::THREADS, B_ALONG_K, PAIRED ? C::TN : 0>;
    static constexpr int PER_STEP = TA::N + TB::N;

    TA ta;
    TB tb;
    MlpOperand A, B;
    int left;                    // steps not requested yet
    int wave, fa[C::FM], fb[C::FN];
    __device__ __forceinline__ void request(char MG_LDS* to) {
        const bool any = left > 0;                       // nothing left: out of range, nothing is read and zeros arrive
        ta.request(to, make_rsrc(A.p, any ? A.bytes : 0u), wave);
        tb.request(to + C::A_BYTES, make_rsrc(B.p, any ? B.bytes : 0u), wave);
        ta.advance(TA::step(A.ld));
        tb.advance(TB::step(B.ld));
        --left;
    }
    __device__ __forceinline__ void read(MlpFragments<C>& f, const char MG_LDS* tile, int s) const {
#pragma unroll
        for (int i = 0; i < C::FM; ++i) f.a[i] = TA::read(tile, TA::further(fa[i], s));
#pragma unroll
        for (int j = 0; j < C::FN; ++j) f.b[j] = TB::read(tile + C::A_BYTES, TB::further(fb[j], s));
    }
    static __device__ __forceinline__ void multiply(MlpSums<C>& sums, const MlpFragments<C>& f) {
#pragma unroll
        for (int i = 0; i < C::FM; ++i)
#pragma unroll
            for (int j = 0; j < C::FN; ++j) sums.v[i][j] = mfma_16x16x32(f.b[j], f.a[i], sums.v[i][j], T());
    }

    // The first STAGES steps requested, the fragments of the first read.  `others` = `first` + one stage.
    __device__ __forceinline__ void start(char MG_LDS* __restrict__ first, char MG_LDS* __restrict__ others, MlpFragments<C>& f, MlpFragments<C>& g) {
        request(first);
#pragma unroll
        for (int s = 1; s < C::STAGES; ++s) request(others + (s - 1) * C::STAGE);
        wait_requests<PER_STEP * (C::STAGES - 1)>();
        step_barrier(first, others);
        read(f, first, 0);
        if constexpr (C::SUBSTEPS == 2) read(g, first, 1);
    }
    // The order of one fragment's worth of instructions, since the compiler, left to itself, issues the reads in a bunch.
    // With one substep: the next fragments' reads between the first half of the multiplications, the requests between all of them
    // (1024 x 3584 outputs, k 2048: 18.9 / 18.5 us, 1024 x 2048, k 3584: 22.2 / 21.5).  LATE, for the second of two substeps: the reads
    // between the second half, no requests.
    template <bool LATE> static __device__ __forceinline__ void interleave() {
        constexpr int M = C::FM * C::FN, H = M / 2, R = C::FM * (A_ALONG_K ? 1 : 2) + C::FN * (B_ALONG_K ? 1 : 2);
#pragma unroll
        for (int i = 0; i < M; ++i) {
            const int at = LATE ? i - H : i, reads = at >= 0 && at < H ? R * (at + 1) / H - R * at / H : 0;
            const int requests = LATE ? 0 : PER_STEP * (i + 1) / M - PER_STEP * i / M;
#pragma unroll
            for (int k = 0; k < reads; ++k) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
            for (int k = 0; k < requests; ++k) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
    }

    // Between two barriers the stage that has arrived, `cur`, is read, and the one before it, which every wave has read,
    // is requested into, `refill`: different stages, so nothing is accessed through both pointers, as they declare.
    // One substep a step: `next` becomes cur's fragments while those of the stage before are multiplied.
    __device__ __forceinline__ void one_substep(const char MG_LDS* __restrict__ cur, char MG_LDS* __restrict__ refill, MlpSums<C>& sums,
                                                const MlpFragments<C>& f, MlpFragments<C>& next) {
        read(next, cur, 0);
        request(refill);
        multiply(sums, f);
        interleave<false>();
    }
    // Two: `g` holds the second fragments of the stage before, and cur's on return; cur's first ones are multiplied in here.
    // The halves are kept apart and the second one's reads late (forward + backward fp16, 2048 tokens, 4096 x 11008, and 1404,
    // 2944 x 5120: 1453 and 384 us; reads where the compiler puts them 1468, 395; nothing kept apart 1552, 393 (bf16); every read early
    // 1474, 382, but 128, 4096 x 11008 268 against 256).
    __device__ __forceinline__ void two_substeps(const char MG_LDS* __restrict__ cur, char MG_LDS* __restrict__ refill, MlpSums<C>& sums,
                                                 MlpFragments<C>& g) {
        MlpFragments<C> f;
        read(f, cur, 0);
        request(refill);
        multiply(sums, g);
        __builtin_amdgcn_sched_barrier(0);
        read(g, cur, 1);
        multiply(sums, f);
        interleave<true>();
    }
    // From one to the next: that has arrived for every wave, and every wave has read all of this one.
    __device__ __forceinline__ void next_stage(char MG_LDS* now, char MG_LDS* next) const {
        wait_requests<PER_STEP * (C::STAGES - 2)>();
        step_barrier(now, next);
    }

    __device__ __forceinline__ void run(MlpShare<C>& share, char MG_LDS* lds, int first, int steps, int m0, int n0, int hidden) {
        const int tid = threadIdx.x, lane = tid & (kWave - 1);
        wave = __builtin_amdgcn_readfirstlane(tid / kWave);
        const int wm = wave % C::WM, wn = wave / C::WM % C::WN, kg = wave / (C::WM * C::WN);
        ta.init(tid, m0, A.ld, 0);
        tb.init(tid, n0, B.ld, hidden);
#pragma unroll
        for (int i = 0; i < C::FM; ++i) fa[i] = TA::fragment(wm * C::TM + i * 16, lane, kg * C::SUBSTEPS);
#pragma unroll
        for (int j = 0; j < C::FN; ++j) fb[j] = TB::fragment(wn * C::TN + j * 16, lane, kg * C::SUBSTEPS);
        MlpSums<C> sums;
#pragma unroll
        for (int i = 0; i < C::FM; ++i)
#pragma unroll
            for (int j = 0; j < C::FN; ++j) sums.v[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        left = steps;
        ta.advance((u32)first * TA::step(A.ld));
        tb.advance((u32)first * TB::step(B.ld));
        MlpFragments<C> f, g;
        start(lds, lds + C::STAGE, f, g);
        const auto after = [](int at) { return at == (C::STAGES - 1) * C::STAGE ? 0 : at + C::STAGE; };
        int at = 0;
        if constexpr (C::SUBSTEPS == 2) {
            multiply(sums, f);
#pragma clang loop unroll(disable)
            for (int k = 1; k < steps; ++k) {
                const int next = after(at);
                next_stage(lds + at, lds + next);
                two_substeps(lds + next, lds + at, sums, g);
                at = next;
            }
            multiply(sums, g);
        } else {   // two sets of fragments in turn; an odd step at the end multiplies zeros
#pragma clang loop unroll(disable)
            for (int k = 0; k < steps; k += 2) {
                const int next = after(at), over = after(next);
                next_stage(lds + at, lds + next);
                one_substep(lds + next, lds + at, sums, f, g);
                next_stage(lds + next, lds + over);
                one_substep(lds + over, lds + next, sums, g, f);
                at = over;
            }
        }
        wait_requests<0>();                              // LDS is used again, by this workgroup or the next
        __syncthreads();
        if constexpr (C::WK == 1) {
#pragma unroll
            for (int i = 0; i < C::FM; ++i)
#pragma unroll
                for (int j = 0; j < C::FN; ++j) share.v[i][j] = sums.v[i][j];
        } else {   // every group hands the others their rows and adds up its own, in the order of the groups
            constexpr int W = C::WM * C::WN, EACH = C::FM / C::WK, HOLDS = C::STAGES * C::STAGE / (W * kWave * 16);
            static_assert(C::FM % C::WK == 0 && HOLDS >= (C::WK - 1) * C::FM * C::FN, "fragments of every wave that LDS holds");
            f32x4 MG_LDS* mine = (f32x4 MG_LDS*)lds + wave % W * kWave + lane;
            // fragment i, j of the rows of group `to`, from group `from`
            const auto place = [&](int to, int from, int i, int j) -> f32x4 MG_LDS& {
                return mine[(((to * (C::WK - 1) + from - (from > to ? 1 : 0)) * EACH + i) * C::FN + j) * (W * kWave)];
            };
#pragma unroll
            for (int from = 0; from < C::WK; ++from)
                if (kg == from) {
#pragma unroll
                    for (int to = 0; to < C::WK; ++to)
#pragma unroll
                        for (int i = 0; i < EACH; ++i)
#pragma unroll
                            for (int j = 0; j < C::FN; ++j) {
                                if (to == from) share.v[i][j] = sums.v[to * EACH + i][j];
                                else place(to, from, i, j) = sums.v[to * EACH + i][j];
                            }
                }
            __syncthreads();
#pragma unroll
            for (int to = 0; to < C::WK; ++to)
                if (kg == to) {
#pragma unroll
                    for (int i = 0; i < EACH; ++i)
#pragma unroll
                        for (int j = 0; j < C::FN; ++j) {
                            f32x4 s = to == 0 ? share.v[i][j] : place(to, 0, i, j);
#pragma unroll
                            for (int from = 1; from < C::WK; ++from) s += from == to ? share.v[i][j] : place(to, from, i, j);
                            share.v[i][j] = s;
                        }
                }
            __syncthreads();
        }
    }
};

// What becomes of the sums.
struct MlpOut { void* out; void* second; const void* in; int M, N; };
constexpr int kMlpStore = 0;     // out [M, N]
constexpr int kMlpPartial = 3;   // out [splits, M, N] in fp32, for mlp_add
constexpr int kMlpGateUp = 1;    // N = hidden: out [M, 2 N] = [gate | up] unless NULL, second [M, N] = silu(gate) * up
constexpr int kMlpActBwd = 2;    // N = hidden: out [M, 2 N] = gradient of `in` [M, 2 N] = [gate | up] for the sums as the gradient of silu(gate) * up

template <typename T>
__device__ __forceinline__ void mlp_store8(rsrc_t r, bool in, u32 at, const float* f) {
    buf_store<4>(r, in ? at * 2u : kNowhere, pack_vec<T, 4>(f));
}
template <typename T>
__device__ __forceinline__ void mlp_load8(float* f, rsrc_t r, bool in, u32 at) {
    unpack_vec<T, 4>(buf_load<4>(r, in ? at * 2u : kNowhere), f);
}

// 16 rows of a wave's tile at a time go through LDS in fp32, so that a lane then has eight consecutive columns and
// eight lanes (four of a 32-column tile) a whole piece of a row: stored straight from the sums, 8 bytes here and there,
// the results take 9 of 33 us at 7168 x 2048 outputs.  N is a multiple of 8.
template <typename T, class C, int WHAT>
__device__ __forceinline__ void mlp_finish(const MlpShare<C>& share, char MG_LDS* lds, const MlpOut& o, int m0, int n0) {
    constexpr bool PAIRED = WHAT == kMlpGateUp;
    constexpr int COLS = PAIRED ? C::TN / 2 : C::TN;     // of the result
    constexpr int LANES = COLS / 8, ROWS = LANES >= 4 ? kWave / LANES : 16, BUFFERS = 2;
    static_assert(C::WAVES * BUFFERS * 16 * C::TN * 4 <= C::STAGE * C::STAGES, "");
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wm = wave % C::WM, wn = wave / C::WM % C::WN, kg = wave / (C::WM * C::WN);
    m0 += wm * C::TM + kg * (C::TM / C::WK);
    const u32 M = (u32)o.M, N = (u32)o.N;
    const rsrc_t out = make_rsrc(o.out, o.out == nullptr ? 0u : M * N * (WHAT == kMlpStore ? 2u : 4u));
    const rsrc_t second = make_rsrc(o.second, PAIRED ? M * N * 2u : 0u);
    const rsrc_t in = make_rsrc(o.in, WHAT == kMlpActBwd ? M * N * 4u : 0u);
    const int row = lane / LANES, unit = lane % LANES * 2;
    const u32 n = (u32)(n0 + wn * COLS + lane % LANES * 8);
    // 16-byte units of a row, permuted by its number: rows of TN floats start in the same bank
    const auto place = [](int r, int u) { return r * C::TN * 4 + ((u ^ (C::TN >= 64 ? r & 15 : (r >> 1) & 7)) << 4); };
    static_assert(C::TN == 128 || C::TN == 64 || C::TN == 32, "");
#pragma unroll
    for (int i = 0; i < C::FM / C::WK; ++i) {
        char MG_LDS* part = lds + (wave * BUFFERS + i % BUFFERS) * (16 * C::TN * 4);
#pragma unroll
        for (int j = 0; j < C::FN; ++j) *(f32x4 MG_LDS*)(part + place(lane & 15, j * 4 + (lane >> 4))) = share.v[i][j];
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += ROWS) {
            const int r = r0 + row;
            const u32 m = (u32)(m0 + i * 16 + r);
            const bool ok = m < M && n < N && r < 16;
            float f[8];
            const auto get = [&](float* to, int u) {
                const f32x4 v = *(const f32x4 MG_LDS*)(part + place(r & 15, u));
#pragma unroll
                for (int q = 0; q < 4; ++q) to[q] = v[q];
            };
            get(f, unit);
            get(f + 4, unit + 1);
            if constexpr (WHAT == kMlpPartial) {
                const u32 at = ok ? (m * N + n) * 4u : kNowhere;
                buf_store<4>(out, at, pack_vec<float, 4>(f));
                buf_store<4>(out, ok ? at + 16u : kNowhere, pack_vec<float, 4>(f + 4));
            } else if constexpr (WHAT == kMlpStore) {
                mlp_store8<T>(out, ok, m * N + n, f);
            } else if constexpr (PAIRED) {
                float u[8], h[8];
                get(u, unit + C::TN / 8);
                get(u + 4, unit + 1 + C::TN / 8);
#pragma unroll
                for (int q = 0; q < 8; ++q) h[q] = (f[q] * fast_sigmoid(f[q])) * u[q];
                mlp_store8<T>(out, ok, m * 2u * N + n, f);
                mlp_store8<T>(out, ok, m * 2u * N + N + n, u);
                mlp_store8<T>(second, ok, m * N + n, h);
            } else {
                float g[8], u[8], dg[8], du[8];
                mlp_load8<T>(g, in, ok, m * 2u * N + n);
                mlp_load8<T>(u, in, ok, m * 2u * N + N + n);
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float s = fast_sigmoid(g[q]);
                    du[q] = f[q] * (g[q] * s);
                    dg[q] = (f[q] * u[q]) * (s * __builtin_fmaf(g[q], 1.0f - s, 1.0f));
                }
                mlp_store8<T>(out, ok, m * 2u * N + n, dg);
                mlp_store8<T>(out, ok, m * 2u * N + N + n, du);
            }
        }
    }
}

// out = the sums of the splits, in their order.  `vectors` of eight elements.
template <typename T>
__global__ void __launch_bounds__(256)
mlp_add(T* __restrict__ out, const float* __restrict__ parts, u32 vectors, int splits) {
    const u32 v = blockIdx.x * 256u + threadIdx.x;
    if (v >= vectors) return;
    const f32x4* at = reinterpret_cast<const f32x4*>(parts) + 2ul * v;
    f32x4 lo = at[0], hi = at[1];
    for (int s = 1; s < splits; ++s) {
        at += 2ul * vectors;
        lo += at[0];
        hi += at[1];
    }
    const float f[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    const Words<4> w = pack_vec<T, 4>(f);
    reinterpret_cast<u32x4*>(out)[v] = u32x4{w.v[0], w.v[1], w.v[2], w.v[3]};
}

// Which tile a workgroup computes.  Workgroups go to the 8 dies round-robin by id: each die gets an equal
// share of consecutive tiles, counted down columns of at most 8 row tiles, so that what it reads through its own
// L2 is a block of both operands of about the same height and width.  The splits of k follow each other.
__device__ __forceinline__ void mlp_tile(int id, int rows, int cols, int splits, int& tm, int& tn, int& split) {
    constexpr int HIGH = 8;
    const int count = rows * cols * splits, die = id % 8, each = count / 8, more = count % 8;
    int t = die * each + (die < more ? die : more) + id / 8;
    split = t / (rows * cols);
    t -= split * rows * cols;
    const int band = t / (HIGH * cols), first = band * HIGH, in = t - first * cols;
    const int h = rows - first < HIGH ? rows - first : HIGH;
    tm = first + in % h;
    tn = in / h;
}

// One product: out from a [M, K] and b [N, K], in `tiles` workgroups (those of all its splits).
struct MlpJob { MlpOperand A, B; MlpOut o; int K, splits, shape; u32 tiles; };

template <typename T, class C, bool A_ALONG_K, bool B_ALONG_K, int WHAT>
__device__ __forceinline__ void mlp_job(const MlpJob& job, u32 id, char MG_LDS* lds) {
    constexpr int BN = WHAT == kMlpGateUp ? C::BN / 2 : C::BN;
    MlpOut o = job.o;
    int tm, tn, split;
    mlp_tile((int)id, (o.M + C::BM - 1) / C::BM, (o.N + BN - 1) / BN, job.splits, tm, tn, split);
    const int steps = (job.K + C::BK - 1) / C::BK, first = split * steps / job.splits, last = (split + 1) * steps / job.splits;
    MlpShare<C> share;
    MlpProduct<T, C, A_ALONG_K, B_ALONG_K, WHAT == kMlpGateUp> p;
    p.A = job.A;
    p.B = job.B;
    p.run(share, lds, first, last - first, tm * C::BM, tn * BN, o.N);
    if constexpr (WHAT == kMlpPartial) o.out = (float*)o.out + (size_t)split * o.M * o.N;
    mlp_finish<T, C, WHAT>(share, lds, o, tm * C::BM, tn * BN);
}

// Workgroups beyond the tiles of a launch read `bytes` from `p` on, which the next launch will want: compute units that have no
// tile bring it into the memory-side cache meanwhile, eight requests a wave at a time so that the tiles are held up little.
// Gate and up / second projection, 1024 tokens, 2048 x 3584: 34.5 / 26.7 -> 35.6 / 22.2 us; 1404, 2944 x 5120 81.7 / 51.4 ->
// 83.5 / 42.0; 300, 2048 x 5504 32.3 / 17.7 -> 34.5 / 14.9.
struct MlpWarm { const void* p; u32 bytes; };
template <class C>
__device__ __forceinline__ void mlp_warm(const MlpWarm& w, u32 id, u32 count, char MG_LDS* lds) {
    constexpr u32 PIECE = C::THREADS * 16;
    const rsrc_t r = make_rsrc(w.p, w.bytes);
    char MG_LDS* to = lds + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * (kWave * 16);
    for (u32 at = id * PIECE; at < w.bytes; at += count * PIECE) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (MG_LDS void*)to, 16, (int)(at + threadIdx.x * 16), 0, 0, 0);
        wait_requests<7>();
    }
    wait_requests<0>();
}

template <typename T, class C, bool A_ALONG_K, bool B_ALONG_K, int WHAT>
__global__ void __launch_bounds__(C::THREADS, C::WAVES / 4)
mlp_gemm(MlpJob job, MlpWarm warm) {
    __shared__ __attribute__((aligned(1024))) char lds[C::STAGE * C::STAGES];
    if (WHAT == kMlpGateUp && blockIdx.x >= job.tiles) return mlp_warm<C>(warm, blockIdx.x - job.tiles, gridDim.x - job.tiles, (char MG_LDS*)lds);
    mlp_job<T, C, A_ALONG_K, B_ALONG_K, WHAT>(job, blockIdx.x, (char MG_LDS*)lds);
}

}  // namespace mg
