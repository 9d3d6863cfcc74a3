// Folded ModDown of hybrid key switching (ckks_keyswitch.cpp:521-673): inverse
// NTT of the P slots, contribution sum_j x_j p_j^-1 - alpha per Q limb (the
// P-side HPS estimate computed once per coefficient), NTT, subtracted from Q.
// The form with the key inner product folded in is mi_moddown_mac.hip.
#include "mi_moddown.hpp"

namespace mi {

constexpr int MODDOWN_TCH = 4;  // target limbs per ModDown-contribution thread

// ---- in-place NTT over a list of polys (limb-major: shared twiddles) ----
struct ListJob {
    u64* p[2 * KS_MAX_ITEMS];
    int npoly, basis0;
    u64 N;
    FastDiv per_limb;  // npoly
    struct View {
        int basis;
        u64* p;
        __device__ u64 load(int i) const { return p[i]; }
        __device__ void store(int i, u64 v) const { p[i] = v; }
    };
    __device__ View view(int k) const {
        const int l = per_limb.div(k), poly = k - l * npoly;
        return View{basis0 + l, p[poly] + (long long)l * N};
    }
    __device__ bool skip(int) const { return false; }
};

struct MdContribArgs {
    const u64* src[2 * KS_MAX_ITEMS];   // P limbs (coefficient domain) of each poly, K limbs apart by N
    u64* tmp;                           // [npoly][L][N]
    const u64* pinv;                    // [L][K]
    int L, K, nq, logN;
    const BasisConst* bc;
};

// One block: 256 coefficients of one poly, up to MODDOWN_TCH target limbs;
// the P-side constants and the targets' p_j^-1 rows are staged in LDS.
template <int K>
__global__ void __launch_bounds__(KS_THREADS) k_moddown_contrib(MdContribArgs a) {
    __shared__ u64 s_pinv[MODDOWN_TCH][K];
    __shared__ u64 s_tq[MODDOWN_TCH], s_ninv[MODDOWN_TCH], s_muhi[MODDOWN_TCH];
    __shared__ u64 s_pq[K];
    __shared__ double s_pinvd[K];
    const u64 N = (u64)1 << a.logN;
    const int poly = blockIdx.y;
    const int t0 = blockIdx.z * MODDOWN_TCH;
    if (t0 >= a.L) return;  // uniform over the block
    const int nt = t0 + MODDOWN_TCH < a.L ? MODDOWN_TCH : a.L - t0;
    for (int e = threadIdx.x; e < nt * K; e += KS_THREADS)
        s_pinv[e / K][e % K] = a.pinv[(long long)(t0 + e / K) * K + e % K];
    if (threadIdx.x < nt) {
        const BasisConst b = a.bc[t0 + threadIdx.x];
        s_tq[threadIdx.x] = b.q;
        s_ninv[threadIdx.x] = b.qninv;
        s_muhi[threadIdx.x] = b.mu_hi;
    }
    if (threadIdx.x >= 64 && threadIdx.x < 64 + K) {
        const BasisConst pb = a.bc[a.nq + threadIdx.x - 64];
        s_pq[threadIdx.x - 64] = pb.q;
        s_pinvd[threadIdx.x - 64] = pb.inv_d;
    }
    __syncthreads();
    // N is a multiple of KS_THREADS: every thread has a coefficient
    const long long i = (long long)blockIdx.x * KS_THREADS + threadIdx.x;
    const u64* src = a.src[poly];
    u64 x[K];
    double est = 0.0;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        x[j] = reduce_4q(src[(long long)j * N + i], s_pq[j]);
        est = __dadd_rn(est, __dmul_rn((double)x[j], s_pinvd[j]));
    }
    u64 al = (u64)__dadd_rn(est, 0.5);
    if (al > (u64)K) al = (u64)K;
    for (int tt = 0; tt < nt; ++tt) {
        U128 acc{0, 0};
#pragma unroll
        for (int j = 0; j < K; ++j) mac128(acc, x[j], s_pinv[tt][j]);  // Montgomery-form p_j^-1
        const u64 q = s_tq[tt];
        const u64 v = redc128_any(acc.lo, acc.hi, q, s_ninv[tt], s_muhi[tt]);
        a.tmp[((long long)poly * a.L + t0 + tt) * N + i] = sub_mod(v, al, q);
    }
}

// forward NTT of the contributions, limb-major (all polys of one modulus together)
struct MdInJob {
    u64* tmp;
    int L, npoly;
    u64 N;
    FastDiv per_limb;  // npoly
    struct View {
        int basis;
        u64* p;
        __device__ u64 load(int i) const { return p[i]; }
        __device__ void store(int i, u64 v) const { p[i] = v; }
    };
    __device__ View view(int k) const {
        const int t = per_limb.div(k), poly = k - t * npoly;
        return View{t, tmp + ((long long)poly * L + t) * N};
    }
    __device__ bool skip(int) const { return false; }
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

void moddown_contrib(const Context& c, int level, int npoly, u64* const* p, u64* T, hipStream_t s) {
    const int L = level + 1, K = c.np;
    const u64 N = c.N;
    MdContribArgs a{};
    for (int k = 0; k < npoly; ++k) a.src[k] = p[k];
    a.tmp = T;
    a.pinv = c.moddown[level].pinv;
    a.L = L;
    a.K = K;
    a.nq = c.nq;
    a.logN = c.logN;
    a.bc = c.d_bc;
    dim3 grid((unsigned)(N / KS_THREADS), npoly, (L + MODDOWN_TCH - 1) / MODDOWN_TCH);
    switch (K) {
#define MI_MODDOWN_CASE(KK) \
        case KK: hipLaunchKernelGGL(k_moddown_contrib<KK>, grid, dim3(KS_THREADS), 0, s, a); break;
        MI_NS_CASES(MI_MODDOWN_CASE)
#undef MI_MODDOWN_CASE
        default: throw Error(-1, "more than 16 special moduli");
    }
    MI_HIP(hipGetLastError());
}

void moddown_contrib_cols(const Context& c, int level, int npoly, u64* T, hipStream_t s) {
    const MdInJob in{T, level + 1, npoly, c.N, fast_div(npoly)};
    launch_pass<true, false>(c, in, npoly * (level + 1), s);
}

static ListJob list_job(const Context& c, int npoly, u64* const* p) {
    ListJob j{};
    for (int k = 0; k < npoly; ++k) j.p[k] = p[k];
    j.npoly = npoly;
    j.per_limb = fast_div(npoly);
    j.basis0 = c.nq;
    j.N = c.N;
    return j;
}

void moddown_p_cols(const Context& c, int npoly, u64* const* p, hipStream_t s) {
    launch_pass<false, false>(c, list_job(c, npoly, p), c.np * npoly, s);
}

void ks_moddown_n(Context& c, int level, int npoly, u64* const* p, const u64* const* base, u64* const* out,
                  u64* T, hipStream_t s) {
    const int L = level + 1, K = c.np;
    const u64 N = c.N;
    if (npoly < 1 || npoly > 2 * KS_MAX_ITEMS) throw Error(-1, "ModDown batch size out of range");
    if (K > MAX_ALPHA) throw Error(-1, "more than 16 special moduli");
    const ListJob j = list_job(c, npoly, p);
    run_ntt_inv(c, j, j, K * npoly, s);
    moddown_contrib(c, level, npoly, p, T, s);
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
    moddown_contrib_cols(c, level, npoly, T, s);
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

}  // namespace mi
