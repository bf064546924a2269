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
// A barrier that accesses through these pointers do not cross: the functions below declare that they do not alias
// (within one step they do not; the compiler would otherwise wait for every request before any LDS read).
__device__ __forceinline__ void step_barrier(const char MG_LDS* a, const char MG_LDS* b, char MG_LDS* c) {
    asm volatile("" ::"s"(a), "s"(b), "s"(c) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::"s"(a), "s"(b), "s"(c) : "memory");
}

template <class C> struct MlpFragments { u32x4 a[C::FM], b[C::FN]; };
template <class C> struct MlpSums { f32x4 v[C::FM][C::FN]; };

// One workgroup's product, bound by LDS: of the 1024 cycles that the matrix instructions of a 256 x 128 x 64 step take, its
// fragments need 1024 (128 bytes a cycle) and its arrival from memory 384, and 1570 are measured with few workgroups,
// 1630 with the chip full.  So the loop keeps all three going: requests are STAGES steps ahead, fragments one
// instruction's worth of k, and one barrier a step serves both the arrival and the reuse of a stage.  What loses: reads and
// multiplications in separate blocks in place of the compiler's own order (33.7 against 31.6 us for 1024 x 7168 outputs,
// k 2048), s_setprio around the multiplications (35.1), waves of 128 x 64 with the k of a step split over two groups (33.4),
// four waves of 128 x 64 (49).
// At 1024 tokens, 2048 x 3584 (bf16, us, these / the library's): gate and up with the activation 30 / 35 + 4, second
// projection 20.1 / 22.3, gradient of h with the activation's 20 / 27 + 8, of x 38.4 / 53, of w3 18.9 / 25.8, of w12 29.4 / 36.
//  `sums.v[i][j][q]` of a wave becomes out[m, n] with
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

    // The first STAGES steps requested, the first fragments of step 0 read.  `others` = `first` + one stage.
    __device__ __forceinline__ void start(char MG_LDS* __restrict__ first, char MG_LDS* __restrict__ others, MlpFragments<C>& f) {
        request(first);
#pragma unroll
        for (int s = 1; s < C::STAGES; ++s) request(others + (s - 1) * C::STAGE);
        wait_requests<PER_STEP * (C::STAGES - 1)>();
        step_barrier(first, others, others);
        read(f, first, 0);
    }
    // One step.  On entry `f` holds its first fragments, read before; on return the next step's.
    __device__ __forceinline__ void step(const char MG_LDS* __restrict__ tile, const char MG_LDS* __restrict__ next, char MG_LDS* __restrict__ refill,
                                         MlpSums<C>& sums, MlpFragments<C>& f) {
        MlpFragments<C> g;
        if constexpr (C::SUBSTEPS == 2) {
            read(g, tile, 1);
            multiply(sums, f);
            f = g;
        }
        wait_requests<PER_STEP * (C::STAGES - 2)>();     // the next step has arrived ...
        step_barrier(tile, next, refill);                // ... for every wave, and every wave has read all of this one
        read(g, next, 0);
        request(refill);
        multiply(sums, f);
        f = g;
    }

    __device__ __forceinline__ void run(MlpSums<C>& sums, char MG_LDS* lds, int K, int m0, int n0, int hidden) {
        const int tid = threadIdx.x, lane = tid & (kWave - 1);
        wave = __builtin_amdgcn_readfirstlane(tid / kWave);
        const int wm = wave % C::WM, wn = wave / C::WM % C::WN, kg = wave / (C::WM * C::WN);
        ta.init(tid, m0, A.ld, 0);
        tb.init(tid, n0, B.ld, hidden);
#pragma unroll
        for (int i = 0; i < C::FM; ++i) fa[i] = TA::fragment(wm * C::TM + i * 16, lane, kg * C::SUBSTEPS);
#pragma unroll
        for (int j = 0; j < C::FN; ++j) fb[j] = TB::fragment(wn * C::TN + j * 16, lane, kg * C::SUBSTEPS);
#pragma unroll
        for (int i = 0; i < C::FM; ++i)
#pragma unroll
            for (int j = 0; j < C::FN; ++j) sums.v[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        const int steps = (K + C::BK - 1) / C::BK;
        left = steps;
        MlpFragments<C> f;
        start(lds, lds + C::STAGE, f);
        int at = 0;
#pragma clang loop unroll(disable)
        for (int k = 0; k < steps; ++k) {
            const int next = at == (C::STAGES - 1) * C::STAGE ? 0 : at + C::STAGE;
            step(lds + at, lds + next, lds + at, sums, f);
            at = next;
        }
        wait_requests<0>();                              // LDS is used again, by this workgroup or the next
        __syncthreads();
        if constexpr (C::WK > 1) {                       // the groups' sums, in order
            constexpr int W = C::WM * C::WN, HOLDS = C::STAGES * C::STAGE / (W * kWave * 16);
            static_assert(HOLDS >= (C::WK - 1) * C::FM * C::FN, "fragments of every wave that LDS holds");
            f32x4 MG_LDS* mine = (f32x4 MG_LDS*)lds + wave % W * kWave + lane;
#pragma unroll
            for (int g = 1; g < C::WK; ++g)
                if (kg == g) {
#pragma unroll
                    for (int i = 0; i < C::FM; ++i)
#pragma unroll
                        for (int j = 0; j < C::FN; ++j) mine[(((g - 1) * C::FM + i) * C::FN + j) * (W * kWave)] = sums.v[i][j];
                }
            __syncthreads();
            if (kg == 0) {
#pragma unroll
                for (int i = 0; i < C::FM; ++i)
#pragma unroll
                    for (int j = 0; j < C::FN; ++j)
#pragma unroll
                        for (int g = 1; g < C::WK; ++g) sums.v[i][j] += mine[(((g - 1) * C::FM + i) * C::FN + j) * (W * kWave)];
            }
            __syncthreads();
        }
    }
};

// What becomes of the sums.
struct MlpOut { void* out; void* second; const void* in; int M, N; };
constexpr int kMlpStore = 0;     // out [M, N]
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
__device__ __forceinline__ void mlp_finish(const MlpSums<C>& sums, char MG_LDS* lds, const MlpOut& o, int m0, int n0) {
    constexpr bool PAIRED = WHAT == kMlpGateUp;
    constexpr int COLS = PAIRED ? C::TN / 2 : C::TN;     // of the result
    constexpr int LANES = COLS / 8, ROWS = LANES >= 4 ? kWave / LANES : 16, BUFFERS = 2;
    static_assert(C::WM * C::WN * BUFFERS * 16 * C::TN * 4 <= C::STAGE * C::STAGES, "");
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wm = wave % C::WM, wn = wave / C::WM % C::WN;
    if (wave >= C::WM * C::WN) return;                   // k groups but the first
    const u32 M = (u32)o.M, N = (u32)o.N;
    const rsrc_t out = make_rsrc(o.out, o.out == nullptr ? 0u : M * N * (WHAT == kMlpStore ? 2u : 4u));
    const rsrc_t second = make_rsrc(o.second, PAIRED ? M * N * 2u : 0u);
    const rsrc_t in = make_rsrc(o.in, WHAT == kMlpActBwd ? M * N * 4u : 0u);
    const int row = lane / LANES, unit = lane % LANES * 2;
    const u32 n = (u32)(n0 + wn * COLS + lane % LANES * 8);
    // 16-byte units of a row, permuted by its number: rows of TN floats start in the same bank
    const auto place = [](int r, int u) { return r * C::TN * 4 + ((u ^ (C::TN == 64 ? r & 15 : (r >> 1) & 7)) << 4); };
    static_assert(C::TN == 64 || C::TN == 32, "");
#pragma unroll
    for (int i = 0; i < C::FM; ++i) {
        char MG_LDS* part = lds + (wave * BUFFERS + i % BUFFERS) * (16 * C::TN * 4);
#pragma unroll
        for (int j = 0; j < C::FN; ++j) *(f32x4 MG_LDS*)(part + place(lane & 15, j * 4 + (lane >> 4))) = sums.v[i][j];
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += ROWS) {
            const int r = r0 + row;
            const u32 m = (u32)(m0 + wm * C::TM + i * 16 + r);
            const bool ok = m < M && n < N && r < 16;
            float f[8];
            const auto get = [&](float* to, int u) {
                const f32x4 v = *(const f32x4 MG_LDS*)(part + place(r & 15, u));
#pragma unroll
                for (int q = 0; q < 4; ++q) to[q] = v[q];
            };
            get(f, unit);
            get(f + 4, unit + 1);
            if constexpr (WHAT == kMlpStore) {
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

// Which tile a workgroup computes.  Workgroups go to the 8 dies round-robin by id: each die gets an equal
// share of consecutive tiles, counted down columns of at most `high` row tiles, so that what it reads through its own
// L2 is a block of both operands of about the same height and width.
__device__ __forceinline__ void mlp_tile(int id, int rows, int cols, int high, int& tm, int& tn) {
    const int count = rows * cols, die = id % 8, each = count / 8, more = count % 8;
    const int t = die * each + (die < more ? die : more) + id / 8;
    const int band = t / (high * cols), first = band * high, in = t - first * cols;
    const int h = rows - first < high ? rows - first : high;
    tm = first + in % h;
    tn = in / h;
}

template <typename T, class C, bool A_ALONG_K, bool B_ALONG_K, int WHAT>
__device__ __forceinline__ void mlp_product(char MG_LDS* lds, int id, const MlpOperand& A, const MlpOperand& B, const MlpOut& o, int K, int high) {
    constexpr int BN = WHAT == kMlpGateUp ? C::BN / 2 : C::BN;
    int tm, tn;
    mlp_tile(id, (o.M + C::BM - 1) / C::BM, (o.N + BN - 1) / BN, high, tm, tn);
    MlpSums<C> sums;
    MlpProduct<T, C, A_ALONG_K, B_ALONG_K, WHAT == kMlpGateUp> p;
    p.A = A;
    p.B = B;
    p.run(sums, lds, K, tm * C::BM, tn * BN, o.N);
    mlp_finish<T, C, WHAT>(sums, lds, o, tm * C::BM, tn * BN);
}

template <typename T, class C, bool A_ALONG_K, bool B_ALONG_K, int WHAT>
__global__ void __launch_bounds__(C::THREADS, C::WAVES / 4)
mlp_gemm(MlpOperand A, MlpOperand B, MlpOut o, int K, int high) {
    __shared__ __attribute__((aligned(1024))) char lds[C::STAGE * C::STAGES];
    mlp_product<T, C, A_ALONG_K, B_ALONG_K, WHAT>((char MG_LDS*)lds, blockIdx.x, A, B, o, K, high);
}

}  // namespace mg
