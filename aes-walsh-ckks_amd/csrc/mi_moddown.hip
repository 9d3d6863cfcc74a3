// Folded ModDown of hybrid key switching (ckks_keyswitch.cpp:521-673): inverse
// NTT of the P slots, contribution sum_j x_j p_j^-1 - alpha per Q limb (the
// P-side HPS estimate summed again for every Q limb: mi_extend.hpp), NTT,
// subtracted from Q.
// The form with the key inner product folded in is mi_moddown_mac.hpp.
#include "mi_extend.hpp"
#include "mi_moddown.hpp"

namespace mi {

// Contributions of the coefficient-domain P limbs to every Q limb, fused with
// the forward column pass.
struct MdExtJob {
    ExtGrid grid;
    const u64* src[2 * KS_MAX_ITEMS];  // K limbs of each poly
    u64* tmp;                          // [npoly][L][N]
    int L;
    u64 N;
    ExtTables t;
    const BasisConst* bc;
    __device__ int targets(int) const { return L; }
    __device__ ExtView view(int poly, int target) const {
        const BasisConst b = bc[target];
        return ExtView{target,
                       src[poly],
                       tmp + ((long long)poly * L + target) * N,
                       (long long)N,
                       t.terms + (long long)target * t.ns,
                       t.src_inv,
                       t.corr + 2 * target,
                       t.ns,
                       t.wide,
                       b.qninv,
                       b.mu_hi};
    }
};

struct MdOutJob {
    const u64* tmp;
    const u64* base[2 * KS_MAX_ITEMS];
    u64* out[2 * KS_MAX_ITEMS];
    int L, npoly;
    u64 N;
    const BasisConst* bc;
    FastDiv per_limb;  // npoly
    struct View {
        int basis;
        const u64* src;
        const u64* base;
        u64* out;
        u64 q;
        double qd, qinv;
        __device__ u64 load(int i) const { return src[i]; }
        __device__ u64 pre(int i) const { return base[i]; }
        __device__ void store_pre(int i, u64 v, u64 b) const { out[i] = sub_mod(b, v, q); }
        __device__ void store_fp(int i, double x, u64 b) const {
            out[i] = FpMod{qd, qinv}.canonical(fp_from_u64(b) - x);
        }
    };
    __device__ View view(int k) const {
        const int t = per_limb.div(k), poly = k - t * npoly;
        return View{t, tmp + ((long long)poly * L + t) * N, base[poly] + (long long)t * N,
                    out[poly] + (long long)t * N, bc[t].q, bc[t].qd, bc[t].inv_d};
    }
    __device__ bool skip(int) const { return false; }
};

void moddown_ext_cols(const Context& c, int level, int npoly, u64* const* p, u64* T, hipStream_t s) {
    MdExtJob j{};
    for (int k = 0; k < npoly; ++k) j.src[k] = p[k];
    j.tmp = T;
    j.L = level + 1;
    j.N = c.N;
    j.t = c.moddown[level];
    j.bc = c.d_bc;
    launch_ext_cols(c, j, npoly, level + 1, s);
}

// The P limbs of npoly polys, a fixed distance apart, as an in-place batch.  They
// run with one limb per workgroup: the tuned plan is measured over the whole
// basis, and these are usually of one kind, for which that form has kernels.
static PlainJob p_limbs(const Context& c, int npoly, u64* const* p) {
    const long long stride = npoly > 1 ? p[1] - p[0] : 0;
    for (int k = 1; k < npoly; ++k)
        if (p[k] - p[k - 1] != stride) throw Error(-1, "ModDown needs evenly spaced P limbs");
    return plain_job(LimbBatch{p[0], stride, c.np, c.nq, c.np * npoly}, c.N);
}

void moddown_p_cols(const Context& c, int npoly, u64* const* p, hipStream_t s) {
    launch_plain_pass(c, false, false, 1, p_limbs(c, npoly, p), c.np * npoly, s);
}

void ks_moddown_n(Context& c, int level, int npoly, u64* const* p, const u64* const* base, u64* const* out,
                  u64* T, hipStream_t s) {
    const int L = level + 1, K = c.np;
    const u64 N = c.N;
    if (npoly < 1 || npoly > 2 * KS_MAX_ITEMS) throw Error(-1, "ModDown batch size out of range");
    if (K > MAX_ALPHA) throw Error(-1, "more than 16 special moduli");
    {
        const PlainJob j = p_limbs(c, npoly, p);
        const long probe = c.probe_open(s, K * npoly);
        launch_plain_pass(c, false, true, 1, j, K * npoly, s);
        launch_plain_pass(c, false, false, 1, j, K * npoly, s);
        c.probe_close(probe, s);
    }
    MdOutJob o{};
    o.tmp = T;
    for (int k = 0; k < npoly; ++k) {
        o.base[k] = base[k];
        o.out[k] = out[k];
    }
    o.L = L;
    o.npoly = npoly;
    o.per_limb = fast_div(npoly);
    o.N = N;
    o.bc = c.d_bc;
    const long probe = c.probe_open(s, npoly * L);
    moddown_ext_cols(c, level, npoly, p, T, s);
    launch_pass<true, true>(c, o, npoly * L, s);
    c.probe_close(probe, s);
}

void ks_moddown(Context& c, int level, u64* p0, u64* p1, const u64* base0, const u64* base1, u64* out0,
                u64* out1, u64* T, hipStream_t s) {
    u64* p[2] = {p0, p1};
    const u64* b[2] = {base0, base1};
    u64* o[2] = {out0, out1};
    ks_moddown_n(c, level, p1 ? 2 : 1, p, b, o, T, s);
}

void ks_moddown_mac(Context& c, int level, int n, const KsItem* items, const u64* D, long long dstride, u64* AP,
                    u64* T, bool montgomery, hipStream_t s, int first, int period) {
    if (period < 1) period = first + n;
    if (n < 1 || n > KS_MAX_ITEMS) throw Error(-1, "key switch batch size out of range");
    if (c.np > MAX_ALPHA) throw Error(-1, "more than 16 special moduli");
    switch (c.parts(level)) {
        case 1: return moddown_mac<1>(c, level, n, items, D, dstride, AP, T, montgomery, s, first, period);
        case 2: return moddown_mac<2>(c, level, n, items, D, dstride, AP, T, montgomery, s, first, period);
        case 3: return moddown_mac<3>(c, level, n, items, D, dstride, AP, T, montgomery, s, first, period);
        default: throw Error(-1, "folded key product takes at most 3 digits");
    }
}

}  // namespace mi
