// RMSNorm backward in one launch, for matrices of few rows: dx and the finished dW, no partial
// rows and no second pass.
#pragma once
#include "mg_device.hpp"

namespace mg {

// Bound by launches and latency, not by bytes: every launch costs 2.4 us of host time, a kernel of
// few rows is one or two round trips to memory, and between pass 1 and the dW reduction lies a
// workspace and a drained chip.  dW[c] = sum_r dy * x * inv_rms does not need the row sum that dx needs, so
// the two are computed side by side by different workgroups of one grid, each reading x and dy once:
// what is read twice is small enough to come from the caches.  Kernel time against pass 1 + reduction
// (us, bf16): 8 x 4096 3.3 / 7.6, 128 x 768 4.3 / 7.8, 512 x 4096 6.3 / 9.6, 1024 x 4096 9.5 / 10.4; fp32 512 x 768
// 4.9 / 7.6.
//   workgroups [0, row_wgs): dx; `wpr` waves share a row (a power of two up to 16), ITEMS vectors per
//     lane, 16 / wpr rows per workgroup;
//   the others, one per 128-byte line of columns: dW; 8 lanes side by side hold the line of a row,
//     128 rows at a time, kRowsInFlight (4: with 8 the workgroup has a compute unit to itself and
//     512 x 4096 takes 7.8 us) of them per thread requested before the first is used; the sums of a
//     wave's 8 rows are added by lane exchanges, those of the 16 waves through LDS, both in a fixed order.
// Rows need no alignment beyond an element's (see RowTail).  Outputs overlap no input (checked on the host):
// a row's dx is written while other workgroups read the row for dW.
//   block = 1024 threads; rows * cols * sizeof(T) < 2^31; ITEMS * 64 * wpr vectors hold a row
constexpr int kSmallBlock = 1024;
constexpr int kRowsInFlight = 4;

template <typename T, int ITEMS>
__global__ void __launch_bounds__(kSmallBlock)
rmsnorm_bwd_small(T* __restrict__ dx, float* __restrict__ dw_f32, T* __restrict__ dw_cast, const T* __restrict__ dy,
                  const T* __restrict__ x, const T* __restrict__ w, const float* __restrict__ inv_rms, int rows, int cols,
                  float inv_cols, int wpr, int row_wgs) {
    constexpr int EPV = 16 / (int)sizeof(T);
    constexpr int WAVES = kSmallBlock / kWave;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid & (kWave - 1);
    const u32 row_bytes = (u32)cols * (u32)sizeof(T);

    if ((int)blockIdx.x < row_wgs) {
        __shared__ float part[WAVES];
        const int slot = wave / wpr;                       // row of the workgroup
        const u32 l = (u32)((wave - slot * wpr) * kWave + lane);   // lane in the row
        const u32 tpr = (u32)wpr * kWave;
        const long row = (long)blockIdx.x * (WAVES / wpr) + slot;
        const bool live = row < rows;
        const long base = live ? row * (long)cols : 0;
        const u32 bytes = live ? row_bytes : 0u;
        const rsrc_t rx = make_rsrc(x + base, bytes), rg = make_rsrc(dy + base, bytes), rd = make_rsrc(dx + base, bytes);
        const rsrc_t rw = make_rsrc(w, row_bytes);
        const float s = live ? inv_rms[row] : 0.0f;
        Words<4> xv[ITEMS], gv[ITEMS], wv[ITEMS];
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const u32 off = (l + i * tpr) * 16u;
            xv[i] = buf_load<4>(rx, off);
            gv[i] = buf_load<4>(rg, off);
            wv[i] = buf_load<4>(rw, off);
        }
        // the half dword that ends a row of an odd number of 2-byte elements
        bool tail[ITEMS];
        const u32 tail_off = row_bytes - 2u;
        const int tail_word = (int)((tail_off & 15u) / 4u);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            tail[i] = sizeof(T) == 2 && (row_bytes & 2u) != 0 && l + i * tpr == tail_off / 16u;
            if (tail[i]) {
                const u32 xb = load_b16<kKeep>(rx, tail_off), gb = load_b16<kKeep>(rg, tail_off), wb = load_b16<kKeep>(rw, tail_off);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (j == tail_word) { xv[i].v[j] = xb; gv[i].v[j] = gb; wv[i].v[j] = wb; }
            }
        }
        float xf[ITEMS][EPV], gw[ITEMS][EPV];
        float a = 0.0f;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            float gf[EPV], wf[EPV];
            unpack_vec<T, 4>(xv[i], xf[i]);
            unpack_vec<T, 4>(gv[i], gf);
            unpack_vec<T, 4>(wv[i], wf);
#pragma unroll
            for (int k = 0; k < EPV; ++k) {
                a = __builtin_fmaf(gf[k] * xf[i][k], wf[k], a);
                gw[i][k] = gf[k] * wf[k];
            }
        }
        a = wave_sum(a);
        if (wpr > 1) {                                     // uniform over the launch
            if (lane == 0) part[wave] = a;
            __syncthreads();
            float t = 0.0f;
            for (int k = 0; k < wpr; ++k) t += part[slot * wpr + k];
            a = t;
        }
        const float c2 = a * (s * s) * s * inv_cols;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            float o[EPV];
#pragma unroll
            for (int k = 0; k < EPV; ++k) o[k] = __builtin_fmaf(gw[i][k], s, -(xf[i][k] * c2));
            const Words<4> v = pack_vec<T, 4>(o);
            buf_store<4>(rd, (l + i * tpr) * 16u, v);
            if (tail[i]) {
                u32 bits = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (j == tail_word) bits = v.v[j];
                __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(bits & 0xffffu), rd, (int)tail_off, 0, kKeep);
            }
        }
        return;
    }

    // ---- dW of one line of columns ----
    __shared__ float sums[WAVES][8 * EPV];
    const u32 c0 = ((u32)blockIdx.x - (u32)row_wgs) * 128u + (u32)(lane & 7) * 16u;   // byte of the row
    const u32 bytes = (u32)rows * row_bytes;
    const rsrc_t rx = make_rsrc(x, bytes), rg = make_rsrc(dy, bytes), rs = make_rsrc(inv_rms, (u32)rows * 4u);
    // a row of an odd number of 2-byte elements ends in half a dword; only that of the last row
    // reaches past the matrix, where the range check drops it
    const bool odd = sizeof(T) == 2 && (row_bytes & 2u) != 0;
    float acc[EPV];
#pragma unroll
    for (int k = 0; k < EPV; ++k) acc[k] = 0.0f;
    for (int r0 = wave * 8 + (lane >> 3); r0 < rows; r0 += kRowsInFlight * 8 * WAVES) {
        Words<4> xv[kRowsInFlight], gv[kRowsInFlight];
        float s[kRowsInFlight];
#pragma unroll
        for (int j = 0; j < kRowsInFlight; ++j) {
            const u32 r = (u32)r0 + (u32)j * (8u * WAVES);
            const u32 off = c0 < row_bytes && r < (u32)rows ? r * row_bytes + c0 : 0xFFFFFFF0u;
            xv[j] = buf_load<4>(rx, off);
            gv[j] = buf_load<4>(rg, off);
            s[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)(r * 4u), 0, 0));
            if (odd && r + 1u == (u32)rows && c0 < row_bytes && row_bytes - c0 <= 16u) {
                const u32 xb = load_b16<kKeep>(rx, bytes - 2u), gb = load_b16<kKeep>(rg, bytes - 2u);
                const u32 word = (row_bytes - 2u - c0) / 4u;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if ((u32)q == word) { xv[j].v[q] = xb; gv[j].v[q] = gb; }
            }
        }
#pragma unroll
        for (int j = 0; j < kRowsInFlight; ++j) {
            float xf[EPV], gf[EPV];
            unpack_vec<T, 4>(xv[j], xf);
            unpack_vec<T, 4>(gv[j], gf);
#pragma unroll
            for (int k = 0; k < EPV; ++k) acc[k] = __builtin_fmaf(gf[k] * xf[k], s[j], acc[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < EPV; ++k) {
        acc[k] += __shfl_xor(acc[k], 8);
        acc[k] += __shfl_xor(acc[k], 16);
        acc[k] += __shfl_xor(acc[k], 32);
    }
    if (lane < 8) {
#pragma unroll
        for (int k = 0; k < EPV; ++k) sums[wave][lane * EPV + k] = acc[k];
    }
    __syncthreads();
    if (tid < 8 * EPV) {
        float t = 0.0f;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) t += sums[k][tid];
        const int c = ((int)blockIdx.x - row_wgs) * 8 * EPV + tid;
        if (c < cols) {
            if (dw_f32 != nullptr) dw_f32[c] = t;
            if (dw_cast != nullptr) Elem<T>::store1(dw_cast + c, t);
        }
    }
}

}  // namespace mg
