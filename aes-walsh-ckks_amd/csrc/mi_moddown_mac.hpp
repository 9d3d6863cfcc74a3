// ModDown with the key inner product folded in, for one number of digits: each
// of mi_moddown_mac{1,2,3}.hip instantiates it, so that they compile side by side.
#pragma once
#include "mi_moddown.hpp"

namespace mi {

// ModDown with the key inner product folded in.
//
// The split form of k_mac (Q slots combined into the outputs, P slots kept
// for ModDown) computed where ModDown reads it: the P slots' products in the
// load of the inverse NTT's first pass, the Q slots' in the store of the
// forward NTT's last pass (with the combine mode, the b term and the
// subtraction of the NTT'd contribution).  The products are neither written
// nor read back.  Each sum holds PARTS <= 3 canonical products (below q
// 2^64: REDC's precondition), reduced once.
// Operands are residues below 4q.
//
// What the keys and moduli are, the same for a whole launch.  Where it is known
// at compile time a thread's 16 products are straight-line code whose loads go
// out together; chosen in the code, each product is a branch of its own and
// waits for its own loads.  N = 2^15, the walsh15 moduli, us, chosen in the code
// / here: rotation at level 1 85.8 / 83.2, one hoisted rotation 69.4 / 59.6.
enum class KeyForm {
    MontBelow61,  // Montgomery-form keys, integer moduli below 2^61
    Mont,         // Montgomery-form keys
    Normal,       // keys in normal form
    Any,          // chosen per product
};
inline KeyForm key_form(const Context& c, bool montgomery) {
    if (!montgomery) return KeyForm::Normal;
    for (const BasisConst& b : c.h_bc)
        if (b.q >= (1ull << 61)) return KeyForm::Mont;
    return KeyForm::MontBelow61;
}
template <KeyForm F>
__device__ __forceinline__ bool form_mont(int mont) {
    return F == KeyForm::Any ? mont != 0 : F != KeyForm::Normal;
}

template <KeyForm F, int PARTS>
__device__ __forceinline__ u64 key_product(const u64* dig, long long dstep, const u64* key, long long kstep, int i,
                                           const BasisConst& b, int mont) {
    U128 s{0, 0};
    if (F == KeyForm::MontBelow61 || (F == KeyForm::Any && b.q < (1ull << 61))) {
        // at most 3 products below 16 q^2: the sum fits in 128 bits and its
        // high word is reduced once, not every operand
#pragma unroll
        for (int d = 0; d < PARTS; ++d) mac128(s, dig[d * dstep + i], key[d * kstep + i]);
    } else {
#pragma unroll
        for (int d = 0; d < PARTS; ++d)
            mac128(s, reduce_4q(dig[d * dstep + i], b.q), reduce_4q(key[d * kstep + i], b.q));
    }
    s.hi = reduce64(s.hi, b.q, b.mu_hi);
    return form_mont<F>(mont) ? redc128(s.lo, s.hi, b.q, b.qninv) : barrett128(s.lo, s.hi, b.q, b.mu_lo, b.mu_hi);
}
// The same as an integer-valued double of magnitude below 3/4 q (Montgomery
// keys; else q/2): moduli below 2^50.
template <KeyForm F, int PARTS>
__device__ __forceinline__ double key_product_fp(const u64* dig, long long dstep, const u64* key, long long kstep,
                                                 int i, const BasisConst& b, int mont) {
    const FpMod m{b.qd, b.inv_d};
    double s = 0.0;
#pragma unroll
    for (int d = 0; d < PARTS; ++d)
        s += m.centred(m.mulq(fp_from_u64(dig[d * dstep + i]), fp_from_u64(key[d * kstep + i])));
    return form_mont<F>(mont) ? m.mul(s, b.rinv_fp, b.rinv_fpq) : m.centred(s);
}

struct KeyProductLists {
    const u64* digits;  // item i's digits at digits + ((first + i) mod period) * dstride: [parts][L+K][N]
    long long dstride;
    int first, period;
    FastDiv per_period;
    const u64* key[KS_MAX_ITEMS];
    int L, K, nq;
    u64 N;
    int mont;  // Montgomery-form keys
    const BasisConst* bc;
    // slot `slot` of poly k (even: a, odd: b) of item k / 2
    __device__ void at(int k, int slot, int basis, const u64*& dig, const u64*& key_p) const {
        const int item = k >> 1, j = first + item;
        dig = digits + (j - per_period.div(j) * period) * dstride + (long long)slot * N;
        key_p = key[item] + ((long long)((k & 1) ? 0 : nq + K) + basis) * N;
    }
};

// inverse NTT first (row) pass over the P slots: load = key product
template <KeyForm F, int PARTS>
struct MacPJob {
    KeyProductLists kp;
    u64* p[2 * KS_MAX_ITEMS];  // poly k's P accumulator (K limbs)
    int npoly;
    FastDiv per_limb;  // npoly
    struct View {
        int basis;
        u64* p;
        const u64* dig;
        const u64* key;
        long long dstep, kstep;
        int mont;
        BasisConst b;
        __device__ u64 load(int i) const { return key_product<F, PARTS>(dig, dstep, key, kstep, i, b, mont); }
        __device__ double load_fp(int i) const { return key_product_fp<F, PARTS>(dig, dstep, key, kstep, i, b, mont); }
        __device__ void store(int i, u64 v) const { p[i] = v; }
    };
    __device__ View view(int k) const {
        const int pi = per_limb.div(k), poly = k - pi * npoly;
        const int basis = kp.nq + pi;
        View v;
        v.basis = basis;
        v.p = p[poly] + (long long)pi * kp.N;
        kp.at(poly, kp.L + pi, basis, v.dig, v.key);
        v.dstep = (long long)(kp.L + kp.K) * kp.N;
        v.kstep = 2LL * (kp.nq + kp.K) * kp.N;
        v.mont = kp.mont;
        v.b = kp.bc[basis];
        return v;
    }
    __device__ bool skip(int) const { return false; }
};

// forward NTT last (row) pass over the Q slots: out = combine(old, key
// product + b term) - NTT(contribution); old and the b term read from a zero
// row where the mode assigns / there is no b term
// MAPPED: items may store through an automorphism.  A form of its own: with the
// map in every switch the 128 switches took 14.8 ms instead of 14.3 and the
// Walsh pairs' relinearisations 40 us more.
template <KeyForm F, int PARTS, bool MAPPED>
struct MdMacOutJob {
    KeyProductLists kp;
    const u64* tmp;                        // [npoly][L][N] NTT'd contributions
    u64* out[2 * KS_MAX_ITEMS];
    const u64* old[2 * KS_MAX_ITEMS];      // out (add mode) or the zero row
    const u64* add[2 * KS_MAX_ITEMS];      // the b term or the zero row
    long long old_step[2 * KS_MAX_ITEMS];  // limb step of old / add: N, or 0 for the zero row
    long long add_step[2 * KS_MAX_ITEMS];
    u32 to[KS_MAX_ITEMS];                  // item's output map: inverse Galois element, or 0
    int npoly, logN;
    FastDiv per_limb;  // npoly
    struct View {
        int basis;
        u32 to;
        int logN;
        const u64* src;
        u64* out;
        const u64* old;
        const u64* add;
        const u64* dig;
        const u64* key;
        long long dstep, kstep;
        int mont;
        BasisConst b;
        __device__ u64 load(int i) const { return src[i]; }
        __device__ u64 pre(int i) const { return add_mod(old[i], add[i], b.q); }
        // An automorphism permutes each row block of the evaluation order into
        // one other block, so mapped stores still fill whole lines.
        __device__ u32 place(int i) const { return MAPPED && to ? galois_index((u32)i, to, logN) : (u32)i; }
        __device__ void store_pre(int i, u64 v, u64 base) const {
            const u64 acc = add_mod(key_product<F, PARTS>(dig, dstep, key, kstep, i, b, mont), base, b.q);
            out[place(i)] = sub_mod(acc, v, b.q);
        }
        __device__ void store_fp(int i, double x, u64 base) const {
            // at most 3/4 q + 5.2q + q < 8q
            const double p = key_product_fp<F, PARTS>(dig, dstep, key, kstep, i, b, mont);
            out[place(i)] = FpMod{b.qd, b.inv_d}.canonical(p - x + fp_from_u64(base));
        }
    };
    __device__ View view(int k) const {
        const int t = per_limb.div(k), poly = k - t * npoly;
        View v;
        v.basis = t;
        v.to = to[poly >> 1];
        v.logN = logN;
        v.src = tmp + ((long long)poly * kp.L + t) * kp.N;
        v.out = out[poly] + (long long)t * kp.N;
        v.old = old[poly] + (long long)t * old_step[poly];
        v.add = add[poly] + (long long)t * add_step[poly];
        kp.at(poly, t, t, v.dig, v.key);
        v.dstep = (long long)(kp.L + kp.K) * kp.N;
        v.kstep = 2LL * (kp.nq + kp.K) * kp.N;
        v.mont = kp.mont;
        v.b = kp.bc[t];
        return v;
    }
    __device__ bool skip(int) const { return false; }
};

template <KeyForm F, int PARTS, bool MAPPED, Arith A = Arith::Both>
void moddown_mac_out(Context& c, int level, int n, const KsItem* items, const KeyProductLists& kp, u64* const* p,
                     u64* T, hipStream_t s) {
    const int L = level + 1, npoly = 2 * n;
    const u64 N = c.N;
    MdMacOutJob<F, PARTS, MAPPED> o{};
    o.kp = kp;
    o.tmp = T;
    for (int i = 0; i < n; ++i) {
        const KsItem& it = items[i];
        if (it.galois && (it.a_mode == 0 || it.b_mode == 0)) throw Error(-1, "a mapped key switch assigns its outputs");
        if (it.galois) {
            // inverse modulo a power of two, by Newton's iteration
            u64 x = it.galois;
            for (int k = 0; k < 5; ++k) x *= 2 - it.galois * x;
            o.to[i] = (u32)(x & (2 * N - 1));
        }
        // poly 2i: a, poly 2i+1: b
        o.out[2 * i] = it.a_out;
        o.out[2 * i + 1] = it.b_out;
        o.old[2 * i] = it.a_mode == 0 ? it.a_out : c.d_zero;
        o.old_step[2 * i] = it.a_mode == 0 ? (long long)N : 0;
        o.old[2 * i + 1] = it.b_mode == 0 ? it.b_out : c.d_zero;
        o.old_step[2 * i + 1] = it.b_mode == 0 ? (long long)N : 0;
        o.add[2 * i] = c.d_zero;
        o.add_step[2 * i] = 0;
        o.add[2 * i + 1] = it.init_b ? it.init_b : c.d_zero;
        o.add_step[2 * i + 1] = it.init_b ? (long long)N : 0;
    }
    o.npoly = npoly;
    o.logN = c.logN;
    o.per_limb = fast_div(npoly);
    const long long probe = c.probe_open(s, npoly * L);
    moddown_ext_cols(c, level, npoly, p, T, s);
    launch_rows_w4<true, A>(c, o, npoly * L, s);
    c.probe_close(probe, s);
}

template <KeyForm F, int PARTS>
void moddown_mac_t(Context& c, int level, int n, const KsItem* items, const u64* D, long long dstride, u64* AP,
                   u64* T, bool montgomery, hipStream_t s, int first, int period) {
    const int K = c.np, npoly = 2 * n;
    const u64 N = c.N;
    KeyProductLists kp{};
    kp.digits = D;
    kp.dstride = dstride;
    kp.first = first;
    kp.period = period;
    kp.per_period = fast_div(period);
    for (int i = 0; i < n; ++i) kp.key[i] = items[i].key;
    kp.L = level + 1;
    kp.K = K;
    kp.nq = c.nq;
    kp.N = N;
    kp.mont = montgomery ? 1 : 0;
    kp.bc = c.d_bc;
    u64* p[2 * KS_MAX_ITEMS];
    for (int i = 0; i < n; ++i) {
        p[2 * i] = AP + (size_t)i * 2 * K * N;
        p[2 * i + 1] = p[2 * i] + (size_t)K * N;
    }
    {
        MacPJob<F, PARTS> in{};
        in.kp = kp;
        for (int k = 0; k < npoly; ++k) in.p[k] = p[k];
        in.npoly = npoly;
        in.per_limb = fast_div(npoly);
        const long long probe = c.probe_open(s, K * npoly);
        launch_rows_w4<false>(c, in, K * npoly, s);
        moddown_p_cols(c, npoly, p, s);
        c.probe_close(probe, s);
    }
    bool mapped = false;
    for (int i = 0; i < n; ++i) mapped = mapped || items[i].galois != 0;
    // Unmapped stores keep the choice where the kernel holds both arithmetics:
    // straight-line, the pass spills 36 to 44 bytes at 128 registers, and 32
    // switches at N = 2^15 took 940 us, not 912.  Integers alone: one switch of one
    // digit at N = 2^14 with the choice 79.1 us, without 76.3.
    if (mapped) moddown_mac_out<F, PARTS, true>(c, level, n, items, kp, p, T, s);
    else if (c.integer_only()) moddown_mac_out<F, PARTS, false, Arith::Int>(c, level, n, items, kp, p, T, s);
    else moddown_mac_out<KeyForm::Any, PARTS, false>(c, level, n, items, kp, p, T, s);
}

template <int PARTS>
void moddown_mac(Context& c, int level, int n, const KsItem* items, const u64* D, long long dstride, u64* AP, u64* T,
                 bool montgomery, hipStream_t s, int first, int period) {
    switch (key_form(c, montgomery)) {
        case KeyForm::MontBelow61:
            return moddown_mac_t<KeyForm::MontBelow61, PARTS>(c, level, n, items, D, dstride, AP, T, montgomery, s, first, period);
        case KeyForm::Mont:
            return moddown_mac_t<KeyForm::Mont, PARTS>(c, level, n, items, D, dstride, AP, T, montgomery, s, first, period);
        default:
            return moddown_mac_t<KeyForm::Normal, PARTS>(c, level, n, items, D, dstride, AP, T, montgomery, s, first, period);
    }
}

}  // namespace mi
