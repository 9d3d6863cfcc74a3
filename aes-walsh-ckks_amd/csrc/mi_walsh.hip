// Walsh S-box product sum: the linear combinations of sign ciphertexts and
// the raw 4+4 products of one output pair, fused into one pass over the
// signs (ckks_walsh_sbox.cpp:984-1043, walsh_sum_for_output_pair, up to its
// relinearisation).
//
// For high mask h = 0..15 and low masks m = 1..15, with integer coefficient
// tables cr, ci ([h][m]; m = 0 is the integer constant V added to b):
//   L(c)  = sum_m c[m] * low_m  (+ V on b)                 (:862-905)
//   Z_h   = L(cr[h]) + pt * L(ci[h])                         (:912-958, pt = encoded i)
//   acc   = Z_0                                               (:999-1005)
//   raw   = sum_{h >= 1} Z_h (x) high_h  (b*b, b*a + a*b, a*a) (:1009-1036)
// Every step is exact arithmetic mod q, so the canonical results equal the
// reference's sequence of scaled additions, plaintext products and tensors.
#include "mi_internal.hpp"
#include "mi_arith.hpp"

#include <cstring>

namespace mi {

constexpr int WALSH_MASKS = 16;

struct WalshArgs {
    const u64* low_b[WALSH_MASKS - 1];  // masks 1..15, L limbs each
    const u64* low_a[WALSH_MASKS - 1];
    const u64* high_b[WALSH_MASKS - 1];
    const u64* high_a[WALSH_MASKS - 1];
    const u64* pt;                      // L limbs, evaluation domain
    u64 *acc_b, *acc_a, *raw_b, *raw_a, *raw_c2;
    // [h][m] as doubles: the high words (a 16-bit integer's low word is zero)
    u32 cr[WALSH_MASKS][WALSH_MASKS];
    u32 ci[WALSH_MASKS][WALSH_MASKS];
    u64 v_lo[2 * WALSH_MASKS], v_hi[2 * WALSH_MASKS];  // |V| of (h, real) at 2h, (h, imag) at 2h+1
    unsigned v_neg;                                     // sign bit per entry
    u64 exact_fp;                                       // bit l: limb l takes the double path
    int logN, pt_mont;
    const BasisConst* bc;
};

__device__ __forceinline__ double walsh_coef(u32 hi) { return __builtin_bit_cast(double, (u64)hi << 32); }

// sum_m c[m] x_m for x_m below q as doubles: exact, the caller has checked
// that the sum of the coefficients' magnitudes times q stays below 2^53.
__device__ __forceinline__ double walsh_lc_fp(const u32* c, const double (&x)[WALSH_MASKS - 1]) {
    double s = walsh_coef(c[1]) * x[0];
#pragma unroll
    for (int m = 2; m < WALSH_MASKS; ++m) s = __builtin_fma(walsh_coef(c[m]), x[m - 1], s);
    return s;
}

// sum_m c[m] x_m mod q for |c| < 2^15 and any q < 2^62, x_m = x1 2^31 + x0
// given as 31-bit halves: each half's sum is below 2^50, exact.  Their
// quotient by q (below 2^19) is estimated in double, off by less than 1/2 and
// a little, and the remainder taken modulo 2^64: in (-q, q), made canonical.
__device__ __forceinline__ u64 walsh_lc(const u32* c, const double (&x0)[WALSH_MASKS - 1],
                                        const double (&x1)[WALSH_MASKS - 1], const BasisConst& b) {
    const double s0 = walsh_lc_fp(c, x0), s1 = walsh_lc_fp(c, x1);
    const double k = __builtin_rint(__builtin_fma(s1, 0x1p31, s0) * b.inv_d);
    // |v| < 2^51 as a 64-bit integer
    auto integer = [](double v) { return __builtin_bit_cast(u64, v + 0x1.8p52) - 0x4338000000000000ull; };
    const u64 r = (integer(s1) << 31) + integer(s0) - integer(k) * b.q;
    return (long long)r < 0 ? r + b.q : r;
}

// A block holds 64 coefficients in 8 waves: side (b or a) x quarter of the
// 16 high masks (quarter 0: h = 0..3, whose h = 0 is the acc term).  A wave
// forms its side of Z_h (b: L(cr) + const + pt L(ci), a: the same without the
// constants) for its 4 masks and the products that side owns:
// b-side Z_b H_b (raw b) and Z_b H_a, a-side Z_a H_b and Z_a H_a (raw c2);
// the partial sums meet in LDS.
constexpr int WALSH_COEFFS = 64;
constexpr int WALSH_BLOCK = 8 * WALSH_COEFFS;

// VALU-bound either way (a coefficient takes 64 linear combinations of 15
// terms and 60 products per limb).  Doubles (moduli small enough for exact
// sums, exact_fp): 15 fused multiply-adds per combination and no reduction,
// six instructions per product.  Integers: the combinations as two sums of
// halves and one double quotient, 128-bit lazy products.  Measured at N = 2^15
// over 36-, 61- and 42-bit limbs, 16 output pairs and their relinearisations:
// 751 us with integer multiply-adds throughout, 583 us.
struct WalshShared {
    u64 cst[2 * WALSH_MASKS];
    u64 part[2][2][4][WALSH_COEFFS];  // [side][product][quarter][coefficient]
};

__device__ __forceinline__ void walsh_fp(const WalshArgs& a, const BasisConst& b, WalshShared& sh, int side,
                                         int quarter, int lane, long long i) {
    const FpMod q{b.qd, b.inv_d};
    double x[WALSH_MASKS - 1];
#pragma unroll
    for (int m = 0; m < WALSH_MASKS - 1; ++m) x[m] = fp_from_u64((side ? a.low_a[m] : a.low_b[m])[i]);
    double pt = q.centred(fp_from_u64(a.pt[i]));
    if (a.pt_mont) pt = q.centred(q.mul(pt, b.rinv_fp, b.rinv_fpq));
    // the rounded 1/q adds at most |x| 2^-53 to a quotient's error: products below 5/2 q
    const double ptq = pt * b.inv_d;
    double s0 = 0.0, s1 = 0.0;
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        const int h = 4 * quarter + k;
        double r = walsh_lc_fp(a.cr[h], x), im = walsh_lc_fp(a.ci[h], x);
        if (side == 0) {
            r += fp_from_u64(sh.cst[2 * h]);
            im += fp_from_u64(sh.cst[2 * h + 1]);
        }
        const double z = q.centred(q.centred(r) + q.mul(im, pt, ptq));
        if (h == 0) {
            (side ? a.acc_a : a.acc_b)[i] = q.canonical(z);
            continue;
        }
        s0 += q.mulq(z, fp_from_u64(a.high_b[h - 1][i]));
        s1 += q.mulq(z, fp_from_u64(a.high_a[h - 1][i]));
    }
    sh.part[side][0][quarter][lane] = q.canonical(s0);
    sh.part[side][1][quarter][lane] = q.canonical(s1);
}

__device__ __forceinline__ void walsh_int(const WalshArgs& a, const BasisConst& b, WalshShared& sh, int side,
                                          int quarter, int lane, long long i) {
    double x0[WALSH_MASKS - 1], x1[WALSH_MASKS - 1];
#pragma unroll
    for (int m = 0; m < WALSH_MASKS - 1; ++m) {
        const u64 x = (side ? a.low_a[m] : a.low_b[m])[i];
        x0[m] = (double)(u32)(x & 0x7fffffffu);
        x1[m] = (double)(u32)(x >> 31);
    }
    const u64 pt = a.pt[i];
    // at most 4 canonical products per 128-bit sum here
    U128 s_h0{0, 0}, s_h1{0, 0};  // side's Z times H_b, times H_a
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        const int h = 4 * quarter + k;
        u64 r = walsh_lc(a.cr[h], x0, x1, b), im = walsh_lc(a.ci[h], x0, x1, b);
        if (side == 0) {
            r = add_mod(r, sh.cst[2 * h], b.q);
            im = add_mod(im, sh.cst[2 * h + 1], b.q);
        }
        const u64 p = a.pt_mont ? mont_mul(im, pt, b.q, b.qninv) : mul_mod(im, pt, b.q, b.mu_lo, b.mu_hi);
        const u64 z = add_mod(r, p, b.q);
        if (h == 0) {
            (side ? a.acc_a : a.acc_b)[i] = z;
            continue;
        }
        mac128(s_h0, z, a.high_b[h - 1][i]);
        mac128(s_h1, z, a.high_a[h - 1][i]);
    }
    sh.part[side][0][quarter][lane] = reduce128(s_h0.lo, s_h0.hi, b.q, b.mu_lo, b.mu_hi);
    sh.part[side][1][quarter][lane] = reduce128(s_h1.lo, s_h1.hi, b.q, b.mu_lo, b.mu_hi);
}

__global__ void __launch_bounds__(WALSH_BLOCK) k_walsh_product_sum(WalshArgs a) {
    __shared__ WalshShared sh;
    const int l = (int)(((long long)blockIdx.x * WALSH_COEFFS) >> a.logN);  // uniform: a block is in one limb
    const int lane = threadIdx.x % WALSH_COEFFS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WALSH_COEFFS);
    const int side = wave >> 2, quarter = wave & 3;
    const long long i = (long long)blockIdx.x * WALSH_COEFFS + lane;
    const BasisConst b = a.bc[l];
    if (threadIdx.x < 2 * WALSH_MASKS) {
        const int t = threadIdx.x;
        const u64 r = reduce128(a.v_lo[t], a.v_hi[t], b.q, b.mu_lo, b.mu_hi);
        sh.cst[t] = ((a.v_neg >> t) & 1) && r ? b.q - r : r;
    }
    __syncthreads();
    if (l < 64 && ((a.exact_fp >> l) & 1)) walsh_fp(a, b, sh, side, quarter, lane, i);
    else walsh_int(a, b, sh, side, quarter, lane, i);
    __syncthreads();
    auto sum4 = [&](int sd, int pr) {
        return add_mod(add_mod(sh.part[sd][pr][0][lane], sh.part[sd][pr][1][lane], b.q),
                       add_mod(sh.part[sd][pr][2][lane], sh.part[sd][pr][3][lane], b.q), b.q);
    };
    if (wave == 0) a.raw_b[i] = sum4(0, 0);                                  // Z_b H_b
    else if (wave == 1) a.raw_a[i] = add_mod(sum4(0, 1), sum4(1, 0), b.q);   // Z_b H_a + Z_a H_b
    else if (wave == 2) a.raw_c2[i] = sum4(1, 1);                            // Z_a H_a
}

void walsh_product_sum(const Context& c, int level, const u64* const* low_b, const u64* const* low_a,
                       const u64* const* high_b, const u64* const* high_a, const short* cr, const short* ci,
                       const u64* v_abs, const int* v_neg, const u64* pt, bool pt_mont, u64* acc_b, u64* acc_a,
                       u64* raw_b, u64* raw_a, u64* raw_c2, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid level");
    WalshArgs a{};
    for (int m = 0; m < WALSH_MASKS - 1; ++m) {
        if (!low_b[m] || !low_a[m] || !high_b[m] || !high_a[m]) throw Error(-1, "null sign ciphertext");
        a.low_b[m] = low_b[m];
        a.low_a[m] = low_a[m];
        a.high_b[m] = high_b[m];
        a.high_a[m] = high_a[m];
    }
    auto high_word = [](short v) {
        const double d = v;
        u64 bits;
        std::memcpy(&bits, &d, 8);
        return (u32)(bits >> 32);
    };
    long long widest = 0;  // largest sum of magnitudes over a row's masks
    for (int h = 0; h < WALSH_MASKS; ++h) {
        long long sr = 0, si = 0;
        for (int m = 0; m < WALSH_MASKS; ++m) {
            const short r = cr[h * WALSH_MASKS + m], im = ci[h * WALSH_MASKS + m];
            if (r == -32768 || im == -32768) throw Error(-1, "coefficient out of range");
            a.cr[h][m] = high_word(r);
            a.ci[h][m] = high_word(im);
            if (m) {
                sr += r < 0 ? -r : r;
                si += im < 0 ? -im : im;
            }
        }
        widest = std::max(widest, std::max(sr, si));
    }
    // a combination and its constant stay below (widest + 1) q
    for (int l = 0; l <= level && l < 64; ++l)
        if (c.h_bc[l].fp && (u64)(widest + 1) <= (1ull << 53) / c.h_bc[l].q) a.exact_fp |= 1ull << l;
    for (int t = 0; t < 2 * WALSH_MASKS; ++t) {
        a.v_lo[t] = v_abs[2 * t];
        a.v_hi[t] = v_abs[2 * t + 1];
        if (v_neg[t]) a.v_neg |= 1u << t;
    }
    a.pt = pt;
    a.pt_mont = pt_mont ? 1 : 0;
    a.acc_b = acc_b;
    a.acc_a = acc_a;
    a.raw_b = raw_b;
    a.raw_a = raw_a;
    a.raw_c2 = raw_c2;
    a.logN = c.logN;
    a.bc = c.d_bc;
    const long long words = (long long)(level + 1) << c.logN;  // a multiple of WALSH_COEFFS
    hipLaunchKernelGGL(k_walsh_product_sum, dim3((unsigned)(words / WALSH_COEFFS)), dim3(WALSH_BLOCK), 0, s, a);
    MI_HIP(hipGetLastError());
}

}  // namespace mi
