// The two projections of the SwiGLU block for a decoding step: out[t, n] = sum_k x[t, k] * w[n, k]
// with at most 64 rows t, and the same with silu(gate) * up folded into the first of them.
#pragma once
#include "mg_device.hpp"

namespace mg {

typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));
typedef half_t f16x8 __attribute__((ext_vector_type(8)));

// D[16 x 16] += A[16 x 32] * B[32 x 16]: lane l holds row l % 16 of A and column l % 16 of B, eight
// consecutive k from 8 * (l / 16) on; of D it holds rows 4 * (l / 16) ... + 3 of column l % 16.
__device__ __forceinline__ f32x4 mfma_16x16x32(u32x4 a, u32x4 b, f32x4 c, bf16_t) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_16x16x32(u32x4 a, u32x4 b, f32x4 c, half_t) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Bound by the stream of the weights: each is used once per call, 16 matrix-instruction columns are
// free next to its load.  What the layout is about is therefore keeping every compute unit on an
// equal share of the weights and the activations out of its way:
//  - one workgroup per compute unit, owning columns [i*N/G, (i+1)*N/G) of the output (PAIRED: the
//    gate row and the up row of each), so that shares differ by one column at most; lanes beyond the
//    share load nothing.  Whole tiles of 8 columns per workgroup leave a last round that is two
//    thirds empty at hidden = 6912: 26.8 against 22.0 us.
//  - MB tiles of 16 weight rows share every activation fragment, and the WAVES waves split K, so
//    the workgroup reads the activations once from L2 (K = 4096, hidden = 6912, 16 tokens: MB = 4
//    22.4 us, 2 26.9, 1 35.5; one token: 21.8).  Waves are added in wave order through LDS.
//  - U steps of 32 per chunk, the next chunk requested before the current one is used, chunks
//    started at a different place in every workgroup (all of them asking for the same lines of
//    the activations at once: 24.9 against 22.0 us).  Weights with the default cache policy: a
//    fragment is half a 128-byte line of each row, and with non-temporal loads the other half is
//    fetched again (25.6 us).
//  - NT tiles of 16 tokens share every weight fragment.  A ring of three to six register buffers instead
//    of two, with buffer loads, is slower (8 tokens 40.6 against 35.2 us for the block): it is not
//    latency that the loop waits for, and lanes of absent tokens, free when masked off, cost with them.
// 113 MB of gate and up weights in 22.0 us = 5.1 TB/s, 57 MB of the second projection (one tile per
// workgroup) in 13.0 us = 4.4 TB/s at 8 tokens; the library products they replace took 28.0 + 24.3
// and the activation between them 4.0.
//   needs: 1 <= tokens <= 16 * NT; K a multiple of 8; 16-byte aligned x and w
//   grid <= N workgroups of WAVES * 64 threads; PAIRED: w holds N gate rows, then N up rows
template <typename T, int MB, int NT, int WAVES, int U, bool PAIRED>
__global__ void __launch_bounds__(WAVES * kWave)
skinny_gemm(T* __restrict__ out, const T* __restrict__ x, const T* __restrict__ w, int tokens, int K, int N) {
    constexpr int TC = PAIRED ? 8 : 16;   // output columns per 16-row tile of weights
    constexpr int COLS = TC * MB;
    constexpr int CHUNK = 32 * U;
    constexpr int PITCH = 20;             // floats per token in the LDS tiles: 16 weight rows and 4 of padding
    __shared__ float part[WAVES][MB][16 * PITCH];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid & (kWave - 1);
    const int r = lane & 15, g = lane >> 4;
    const int lo = (int)((long)blockIdx.x * N / gridDim.x);
    const int hi = (int)((long)(blockIdx.x + 1) * N / gridDim.x);

    const T* xp[NT];                      // rows r, r + 16, ... of the activations
    bool x_mine[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        x_mine[t] = t * 16 + r < tokens;
        xp[t] = x + (x_mine[t] ? (long)(t * 16 + r) * K : 0L) + g * 8;
    }
    const int chunks = K / CHUNK;
    const int n = chunks > wave ? (chunks - wave + WAVES - 1) / WAVES : 0;   // chunks wave, wave + WAVES, ...
    const int skew = n > 0 ? (int)(blockIdx.x / 8u * 5u) % n : 0;            // / 8: the XCDs have an L2 each

    for (int n0 = lo; n0 < hi; n0 += COLS) {
        const T* wp[MB];
        bool w_mine[MB];
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            const int col = n0 + m * TC + (r & (TC - 1));
            w_mine[m] = col < hi;
            const long row = (w_mine[m] ? col : lo) + (PAIRED && r >= 8 ? (long)N : 0L);
            wp[m] = w + row * K + g * 8;
        }
        f32x4 acc[MB][NT];
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

        struct Fragments { u32x4 w[MB][U]; u32x4 x[NT][U]; };
        auto load = [&](Fragments& f, int i) {
            int j = i + skew;
            if (j >= n) j -= n;
            const int k = (wave + j * WAVES) * CHUNK;
#pragma unroll
            for (int m = 0; m < MB; ++m) {
#pragma unroll
                for (int u = 0; u < U; ++u) f.w[m][u] = u32x4{0, 0, 0, 0};
                if (w_mine[m]) {
#pragma unroll
                    for (int u = 0; u < U; ++u) f.w[m][u] = *reinterpret_cast<const u32x4*>(wp[m] + k + u * 32);
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int u = 0; u < U; ++u) f.x[t][u] = u32x4{0, 0, 0, 0};
                if (x_mine[t]) {
#pragma unroll
                    for (int u = 0; u < U; ++u) f.x[t][u] = *reinterpret_cast<const u32x4*>(xp[t] + k + u * 32);
                }
            }
        };
        auto use = [&](const Fragments& f) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[m][t] = mfma_16x16x32(f.w[m][u], f.x[t][u], acc[m][t], T());
        };
        Fragments f0, f1;
        if (n > 0) load(f0, 0);
        for (int i = 0; i < n; i += 2) {
            if (i + 1 < n) load(f1, i + 1);
            use(f0);
            if (i + 1 < n) {
                if (i + 2 < n) load(f0, i + 2);
                use(f1);
            }
        }
        // the rest of K in steps of 32, the last one possibly short (zeros on both sides)
        for (int k = chunks * CHUNK + wave * 32; k < K; k += WAVES * 32) {
            const bool in = k + g * 8 < K;
            u32x4 xv[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                xv[t] = u32x4{0, 0, 0, 0};
                if (in && x_mine[t]) xv[t] = *reinterpret_cast<const u32x4*>(xp[t] + k);
            }
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                u32x4 wv = {0, 0, 0, 0};
                if (in && w_mine[m]) wv = *reinterpret_cast<const u32x4*>(wp[m] + k);
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[m][t] = mfma_16x16x32(wv, xv[t], acc[m][t], T());
            }
        }

        // the waves' sums, one tile of 16 tokens after the other through the same LDS
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
            if (tt > 0 || n0 != lo) __syncthreads();   // the previous sums have been read
#pragma unroll
            for (int m = 0; m < MB; ++m) *reinterpret_cast<f32x4*>(&part[wave][m][r * PITCH + g * 4]) = acc[m][tt];
            __syncthreads();
            for (int i = tid; i < 16 * COLS; i += WAVES * kWave) {
                const int c = i % COLS, t = i / COLS;
                const int at = t * PITCH + c % TC;
                float s = 0.0f, up = 0.0f;
#pragma unroll
                for (int q = 0; q < WAVES; ++q) {
                    s += part[q][c / TC][at];
                    if constexpr (PAIRED) up += part[q][c / TC][at + 8];
                }
                if constexpr (PAIRED) s = (s * fast_sigmoid(s)) * up;
                if (tt * 16 + t < tokens && n0 + c < hi) Elem<T>::store1(out + (long)(tt * 16 + t) * N + n0 + c, s);
            }
        }
    }
}

}  // namespace mg
