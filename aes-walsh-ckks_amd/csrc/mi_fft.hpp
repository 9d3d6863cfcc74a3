// The special FFTs of encoding (decimation in frequency) and decoding
// (decimation in time) in two launches instead of one per stage: a stage is
// under 3 us of work at any ring dimension, so the logN launches were what one
// took.  The stages with pairs up to FFT_BLOCK/2 apart run in LDS, a contiguous
// block of FFT_BLOCK points per workgroup; the others in registers, one thread
// per column of N / FFT_BLOCK points FFT_BLOCK apart.  Each butterfly is the
// single-stage form's separately rounded IEEE operations on the same operands,
// so the results are the same bit for bit.
#pragma once
#include "mi_internal.hpp"

namespace mi {

constexpr int FFT_BLOCK = 2048;  // 32 KB of LDS
constexpr int FFT_THREADS = 256;

struct C64 {
    double re, im;
};

// DIF: x0 = u + v, x1 = (u - v) w.  DIT: x0 = u + v w, x1 = u - v w.
template <bool DIF>
__device__ __forceinline__ void fft_butterfly(C64& u, C64& v, const C64& w) {
    if constexpr (DIF) {
        const C64 s{__dadd_rn(u.re, v.re), __dadd_rn(u.im, v.im)};
        const double dr = __dsub_rn(u.re, v.re), di = __dsub_rn(u.im, v.im);
        v = C64{__dsub_rn(__dmul_rn(dr, w.re), __dmul_rn(di, w.im)), __dadd_rn(__dmul_rn(dr, w.im), __dmul_rn(di, w.re))};
        u = s;
    } else {
        const C64 t{__dsub_rn(__dmul_rn(v.re, w.re), __dmul_rn(v.im, w.im)),
                    __dadd_rn(__dmul_rn(v.re, w.im), __dmul_rn(v.im, w.re))};
        v = C64{__dsub_rn(u.re, t.re), __dsub_rn(u.im, t.im)};
        u = C64{__dadd_rn(u.re, t.re), __dadd_rn(u.im, t.im)};
    }
}

// Stages k = 1 .. 2^logb / 2 of blockIdx.y's transform (pairs k apart, group i
// of N / 2k with twiddle tw[N / 2k + i]); `in(j)` gives point j.
template <bool DIF, class IN>
__global__ void __launch_bounds__(FFT_THREADS)
k_fft_block(IN in, C64* __restrict__ x, const C64* __restrict__ tw, int logN, int logb) {
    __shared__ C64 s[FFT_BLOCK];
    const int B = 1 << logb, base = blockIdx.x << logb;
    C64* out = x + ((long long)blockIdx.y << logN);
    for (int j = threadIdx.x; j < B; j += FFT_THREADS) s[j] = in(blockIdx.y, base + j);
    __syncthreads();
    for (int st = 0; st < logb; ++st) {
        const int lk = DIF ? st : logb - 1 - st, k = 1 << lk;
        const int first = (1 << (logN - 1 - lk)) + (base >> (lk + 1));  // twiddle of the block's group 0
        for (int t = threadIdx.x; t < B / 2; t += FFT_THREADS) {
            const int i = t >> lk, a = (i << (lk + 1)) + (t & (k - 1));
            C64 u = s[a], v = s[a + k];
            fft_butterfly<DIF>(u, v, tw[first + i]);
            s[a] = u;
            s[a + k] = v;
        }
        __syncthreads();
    }
    for (int j = threadIdx.x; j < B; j += FFT_THREADS) out[base + j] = s[j];
}

// The remaining R stages: 2^R points FFT_BLOCK apart per thread.
template <bool DIF, int R>
__global__ void __launch_bounds__(FFT_THREADS) k_fft_cols(C64* __restrict__ x, const C64* __restrict__ tw) {
    C64* col = x + ((long long)blockIdx.y << R) * FFT_BLOCK + blockIdx.x * FFT_THREADS + threadIdx.x;
    C64 v[1 << R];
#pragma unroll
    for (int t = 0; t < (1 << R); ++t) v[t] = col[(long long)t * FFT_BLOCK];
#pragma unroll
    for (int st = 0; st < R; ++st) {
        const int lk = DIF ? st : R - 1 - st, k = 1 << lk;
#pragma unroll
        for (int t = 0; t < (1 << R); ++t) {
            if (t & k) continue;
            fft_butterfly<DIF>(v[t], v[t + k], tw[(1 << (R - 1 - lk)) + (t >> (lk + 1))]);
        }
    }
#pragma unroll
    for (int t = 0; t < (1 << R); ++t) col[(long long)t * FFT_BLOCK] = v[t];
}

// `count` transforms of 2^logN points at x; the first pass reads `in`, the
// second what the first wrote.
template <bool DIF>
void launch_fft_cols(C64* x, const C64* tw, int logN, int count, hipStream_t s) {
    const dim3 g(FFT_BLOCK / FFT_THREADS, count), b(FFT_THREADS);
    switch (logN) {
        case 12: hipLaunchKernelGGL((k_fft_cols<DIF, 1>), g, b, 0, s, x, tw); break;
        case 13: hipLaunchKernelGGL((k_fft_cols<DIF, 2>), g, b, 0, s, x, tw); break;
        case 14: hipLaunchKernelGGL((k_fft_cols<DIF, 3>), g, b, 0, s, x, tw); break;
        case 15: hipLaunchKernelGGL((k_fft_cols<DIF, 4>), g, b, 0, s, x, tw); break;
        case 16: hipLaunchKernelGGL((k_fft_cols<DIF, 5>), g, b, 0, s, x, tw); break;
        default: return;  // the block is the whole transform
    }
    MI_HIP(hipGetLastError());
}
template <bool DIF, class IN>
void launch_fft_block(const IN& in, C64* x, const C64* tw, int logN, int count, hipStream_t s) {
    const int logb = logN < 11 ? logN : 11;
    hipLaunchKernelGGL((k_fft_block<DIF, IN>), dim3(1u << (logN - logb), count), dim3(FFT_THREADS), 0, s, in, x, tw,
                       logN, logb);
    MI_HIP(hipGetLastError());
}

}  // namespace mi
