// Base extension fused into the forward column pass.
//
// The HPS extension (ckks_keyswitch.cpp:278-332, 521-673) of a digit's or of
// the P limbs' coefficients x_0..x_{ns-1} to a target modulus m is
//   sum_i x_i c_i - alpha Q mod m,   alpha = round(sum_i x_i / q_i),
// followed by the target limb's forward NTT.  Here the column pass of that NTT
// forms its own input: a thread runs over the sources and, for its 16
// positions, over the words of each.  Nothing is written between the extension
// and the transform, and the workgroups of one block of columns follow each
// other over all targets on one XCD (workgroups are dealt round robin), so the
// sources come from memory once and from that XCD's L2 for the other targets.
// The estimate alpha is summed per target instead of once per eight: 4
// instructions a source against the 16 bytes a word that the separate kernel
// wrote and this pass read back.
#pragma once
#include "mi_ntt_kernels.hpp"

namespace mi {

// One limb of an extension's output, as a View of a column pass.
struct ExtView {
    int basis;
    const u64* src;  // ns limbs of N coefficients, canonical
    u64* out;
    long long N;
    const ExtTerm* terms;
    const double* src_inv;
    const u64* corr;
    int ns;
    u64 wide;  // bit i: source i has 50 bits or more
    u64 qninv, mu_hi;
    static constexpr bool BLOCK = true;
    __device__ void store(int i, u64 v) const { out[i] = v; }

    // Target below 2^50.  A source below 2^50 enters as a double, a wider one as
    // two 32-bit halves with the constants c_i and 2^32 c_i; each product is at
    // most 5/8 m (one or two of 1/2 m and a little), so four sources add 4 m
    // and the sum is centred after every four.
    template <class AT>
    __device__ __forceinline__ void load_block(const BfFp& bf, AT at, u64 (&x)[E]) const {
        const FpMod& m = bf.m;
        double est[E], acc[E];
#pragma unroll
        for (int j = 0; j < E; ++j) est[j] = acc[j] = 0.0;
        for (int i = 0; i < ns; ++i) {
            const u64* s = src + (long long)i * N;
            const ExtTerm t = terms[i];
            const double inv = src_inv[i];
            const double c = BfFp::d(t.v[0]), cq = BfFp::d(t.v[1]);
            u64 v[E];
#pragma unroll
            for (int j = 0; j < E; ++j) v[j] = s[at(j)];
            if ((wide >> i) & 1) {
                const double ch = BfFp::d(t.v[2]), chq = BfFp::d(t.v[3]);
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    const double hi = (double)(u32)(v[j] >> 32), lo = (double)(u32)v[j];
                    // hi 2^32 + lo in one rounding: (double)v
                    est[j] = __dadd_rn(est[j], __dmul_rn(__builtin_fma(hi, 0x1p32, lo), inv));
                    acc[j] += m.mul(lo, c, cq) + m.mul(hi, ch, chq);
                }
            } else {
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    const double d = fp_from_u64(v[j]);
                    est[j] = __dadd_rn(est[j], __dmul_rn(d, inv));
                    acc[j] += m.mul(d, c, cq);
                }
            }
            if ((i & 3) == 3) {
#pragma unroll
                for (int j = 0; j < E; ++j) acc[j] = m.centred(acc[j]);
            }
        }
        const double Q = BfFp::d(corr[0]), Qq = BfFp::d(corr[1]), top = (double)ns;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const double a = __builtin_floor(__dadd_rn(est[j], 0.5));
            x[j] = BfFp::u(m.centred(acc[j] - m.mul(a < top ? a : top, Q, Qq)));
        }
    }

    // Any target: exact 128-bit sums of at most 16 products (< 2^128), the
    // constants in Montgomery form, one REDC.  Eight positions at a time: a
    // sum takes four registers.  The next source's words and constants are
    // loaded before this one's are used.  A word becomes a double for the
    // estimate as hi 2^32 + lo in one rounding, which is (double)v.
    template <class AT>
    __device__ __forceinline__ void load_block(const BfInt& bf, AT at, u64 (&x)[E]) const {
        const u64 q = bf.q;
        // ns products below 2^50 m, or 4 below 2^62 m, stay below 2^64 m
        const bool reduced = wide == 0 || ns <= 4;
        const u64 Q = corr[0], Qs = corr[1];
#pragma unroll
        for (int h = 0; h < E; h += E / 2) {
            double est[E / 2];
            U128 acc[E / 2];
#pragma unroll
            for (int j = 0; j < E / 2; ++j) {
                est[j] = 0.0;
                acc[j] = U128{0, 0};
            }
            u64 next[E / 2], next_c = terms[0].v[0];
            double next_inv = src_inv[0];
#pragma unroll
            for (int j = 0; j < E / 2; ++j) next[j] = src[at(h + j)];
            for (int i = 0; i < ns; ++i) {
                const int n = i + 1 < ns ? i + 1 : i;
                const u64* s = src + (long long)n * N;
                const u64 c = next_c;
                const double inv = next_inv;
                u64 v[E / 2];
#pragma unroll
                for (int j = 0; j < E / 2; ++j) v[j] = next[j];
#pragma unroll
                for (int j = 0; j < E / 2; ++j) next[j] = s[at(h + j)];
                next_c = terms[n].v[0];
                next_inv = src_inv[n];
#pragma unroll
                for (int j = 0; j < E / 2; ++j) {
                    const double d = __builtin_fma((double)(u32)(v[j] >> 32), 0x1p32, (double)(u32)v[j]);
                    est[j] = __dadd_rn(est[j], __dmul_rn(d, inv));
                    mac128(acc[j], v[j], c);
                }
            }
#pragma unroll
            for (int j = 0; j < E / 2; ++j) {
                u64 al = (u64)__dadd_rn(est[j], 0.5);
                if (al > (u64)ns) al = (u64)ns;
                const u64 hi = reduced ? acc[j].hi : reduce64(acc[j].hi, q, mu_hi);
                x[h + j] = sub_mod(redc128(acc[j].lo, hi, q, qninv), shoup(al, Q, Qs, q), q);
            }
        }
    }
};

// Block b of a launch over `tiles` column blocks (of one source each) and up
// to `targets` limbs: the targets of a tile consecutive on one XCD.
struct ExtGrid {
    int tiles, targets;
    FastDiv per_tile;  // targets
    __device__ __forceinline__ bool locate(int b, int& tile, int& target) const {
        const int local = b >> 3, tl = per_tile.div(local);
        target = local - tl * targets;
        tile = tl * 8 + (b & 7);
        return tile < tiles;
    }
};

// A: Both, or Int for contexts whose moduli are all integers, held to three
// waves per SIMD (164 registers).  Both takes 214 registers and two waves,
// which suits the doubles (16 words in flight) but made integer key switches
// slower than the separate extension had been.  N = 2^16, 30 + 10 limbs of 60
// bits, us, separate / two waves / three: hoist 131 / 140 / 132, one key switch
// 285 / 297 / 283, four 917 / 960 / 909, 32 7094 / 7230 / 6931.
template <int LOGN, Arith A, class Job>
__global__ void __launch_bounds__(NTT_THREADS) __attribute__((amdgpu_waves_per_eu(A == Arith::Int ? 3 : 1)))
k_ext_cols(NttTabs tb, Job job) {
    constexpr int n1 = LOGN / 2, wpl = pass_wpl(n1, LOGN - n1);
    __shared__ u64 lds[NTT_LDS_WORDS];
    int tile, target;
    if (!job.grid.locate(blockIdx.x, tile, target)) return;
    const int source = tile / wpl;  // wpl is a power of two
    if (target >= job.targets(source)) return;
    const ExtView v[1] = {job.view(source, target)};
    const bool live[1] = {true};
    const int w = tile - source * wpl;
    if constexpr (A == Arith::Both) {
        if (tb.fp(v[0].basis)) {
            pass_body<LOGN, true, false, 1, BfFp>(tb, v, live, w, lds);
            return;
        }
    }
    pass_body<LOGN, true, false, 1, BfInt>(tb, v, live, w, lds);
}

// Launches the fused extension and column pass of `sources` sources with up to
// `targets` target limbs each (job.grid is set here).
template <class Job>
void launch_ext_cols(const Context& c, Job job, int sources, int targets, hipStream_t s) {
    const NttTabs tb = tabs_of(c);
    const bool integer = c.integer_only();
#define MI_EXT(LN)                                                                                    \
    {                                                                                                 \
        job.grid = ExtGrid{sources * pass_wpl(LN / 2, LN - LN / 2), targets, fast_div(targets)};      \
        const long long blocks = (long long)((job.grid.tiles + 7) / 8) * 8 * targets;                 \
        if (blocks >= (8LL << 20)) throw Error(-1, "base extension: too many limbs in one launch");   \
        const dim3 g((unsigned)blocks), b(pass_threads(LN / 2, LN - LN / 2));                         \
        if (integer) hipLaunchKernelGGL((k_ext_cols<LN, Arith::Int, Job>), g, b, 0, s, tb, job);      \
        else hipLaunchKernelGGL((k_ext_cols<LN, Arith::Both, Job>), g, b, 0, s, tb, job);             \
    }
    MI_NTT_LOGN_CASES(MI_EXT)
#undef MI_EXT
    MI_HIP(hipGetLastError());
}

}  // namespace mi
