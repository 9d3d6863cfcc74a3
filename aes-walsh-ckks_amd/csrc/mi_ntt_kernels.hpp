// NTT pass kernels templated on a Job (see mi_ntt.hip).
//
// A Job is a trivially copyable struct with
//   __device__ View view(int k) const;   // limb k of the batch
//   __device__ bool skip(int k) const;   // whole limb skipped (uniform)
// and a View with
//   int basis;                            // basis index of the limb
//   __device__ u64 load(int i) const;     // coefficient / slot i
//   __device__ void store(int i, u64 v) const;
// A View may also offer `u64 pre(int i) const` and
// `void store_pre(int i, u64 v, u64 pre) const`: the pass then reads pre(i)
// for its output positions together with its input, before the butterflies,
// and stores through store_pre, so an output that combines the transform
// with another operand does not wait for that operand's loads at the end.
// For limbs in double arithmetic (BasisConst::fp) a View of a first pass may
// offer `double load_fp(int i) const`, its input as an integer-valued double
// below q in magnitude, and a View of a forward transform's second pass
// `void store_fp(int i, double x, u64 pre) const` (`pre` as above, else 0),
// which takes the transform's output x before it is made canonical
// (|x| < 5.2q) and stores the canonical result.
// A View with `static constexpr bool BLOCK` forms all E inputs of a thread in
// one call, load_block(arithmetic, positions, x), in the working form.  A View
// of an inverse transform's second pass may name its own `const u64* inv_scale`
// in place of BasisConst::inv_last.
// Forward column pass: load = job input, store = intermediate.
// Forward row pass: load = intermediate, store = canonical output.
// Inverse row pass: load = input (canonical), store = intermediate.
// Inverse column pass: load = intermediate, store = canonical output.
// The intermediate is in the working form of the limb's modulus (lazy residues
// or doubles, mi_ntt_core.hpp): the two passes only hand it to each other.
#pragma once
#include <type_traits>
#include "mi_internal.hpp"
#include "mi_ntt_core.hpp"

namespace mi {

struct NttTabs {
    const u64* fwd;
    const u64* fwd_shoup;
    const u64* inv;
    const u64* inv_shoup;
    const BasisConst* bc;
    u64 N;
    // BasisConst::fp of the first 128 basis indices as kernel arguments: the
    // choice of the arithmetic comes before the first data load and must not
    // wait for a table (reading it from bc cost the 60-bit batch 2 %).
    u64 fp_mask[2];
    __device__ __forceinline__ bool fp(int basis) const {
        if (basis >= 128) return bc[basis].fp != 0;
        return ((basis < 64 ? fp_mask[0] : fp_mask[1]) >> (basis & 63)) & 1;
    }
};

inline NttTabs tabs_of(const Context& c) {
    NttTabs t{c.d_fwd, c.d_fwd_shoup, c.d_inv, c.d_inv_shoup, c.d_bc, c.N, {0, 0}};
    for (int b = 0; b < c.nb() && b < 128; ++b)
        if (c.h_bc[b].fp) t.fp_mask[b >> 6] |= 1ull << (b & 63);
    return t;
}

// In-place NTT over a strided batch.  Workgroups walk the batch modulus-major
// (all polys' limb 0, then limb 1, ...): the workgroups resident on one XCD
// at a time then share a single modulus's twiddle tables in that XCD's L2.
struct PlainJob {
    LimbBatch b;
    u64 N;
    int npolys;        // polys per modulus: b.count / b.lpp
    FastDiv per_limb;  // npolys
    struct View {
        int basis;
        u64* p;
        __device__ u64 load(int i) const { return p[i]; }
        __device__ void store(int i, u64 v) const { p[i] = v; }
    };
    __device__ View view(int k) const {
        const int l = per_limb.div(k), poly = k - l * npolys;
        return View{b.basis0 + l, b.base + (long long)poly * b.stride + (long long)l * N};
    }
    __device__ bool skip(int) const { return false; }
};
inline PlainJob plain_job(const LimbBatch& b, u64 N) {
    return PlainJob{b, N, b.count / b.lpp, fast_div(b.count / b.lpp)};
}

// Pass geometry, fixed at compile time by log2 N: n1 = n/2 column stages and
// n2 = n - n1 row stages.  A pass whose groups have 2^logr elements and which
// has 2^logother groups per limb runs workgroups of pass_threads() threads
// holding pass_groups() groups, pass_wpl() workgroups per limb.
constexpr int pass_threads(int logr, int logother) {
    return ((1 << (logr - LOGE)) << logother) > NTT_THREADS ? NTT_THREADS : ((1 << (logr - LOGE)) << logother);
}
constexpr int pass_groups(int logr, int logother) { return pass_threads(logr, logother) >> (logr - LOGE); }
constexpr int pass_wpl(int logr, int logother) { return (1 << logother) / pass_groups(logr, logother); }

template <class V, class = void>
struct HasPre : std::false_type {};
template <class V>
struct HasPre<V, std::void_t<decltype(&V::pre)>> : std::true_type {};
template <class V, class = void>
struct HasLoadFp : std::false_type {};
template <class V>
struct HasLoadFp<V, std::void_t<decltype(&V::load_fp)>> : std::true_type {};
template <class V, class = void>
struct HasBlock : std::false_type {};
template <class V>
struct HasBlock<V, std::void_t<decltype(V::BLOCK)>> : std::true_type {};
template <class V, class = void>
struct HasInvScale : std::false_type {};
template <class V>
struct HasInvScale<V, std::void_t<decltype(&V::inv_scale)>> : std::true_type {};
template <class V, class = void>
struct HasStoreFp : std::false_type {};
template <class V>
struct HasStoreFp<V, std::void_t<decltype(&V::store_fp)>> : std::true_type {};

// LPB limbs per workgroup (1 or 2): workgroup b serves limbs LPB*(b / wpl) +
// 0..LPB-1 of a launch over `count` limbs; a limb past `count` or skipped by
// the job is left alone (uniform over the workgroup).
template <int LPB, class Job, class V>
__device__ __forceinline__ bool limb_views(const Job& job, int first, int count, V (&v)[LPB], bool (&live)[LPB]) {
    bool any = false;
    int k0 = -1;
#pragma unroll
    for (int i = 0; i < LPB; ++i) {
        const int k = first + i;
        live[i] = k < count && !job.skip(k);
        if (live[i] && k0 < 0) k0 = k;
        any = any || live[i];
    }
    if (!any) return false;
#pragma unroll
    for (int i = 0; i < LPB; ++i) v[i] = job.view(live[i] ? first + i : k0);  // a dead limb borrows a live view
    return true;
}

// One pass over the LPB limbs of a workgroup in the arithmetic BF (all of
// them; see mi_ntt_core.hpp).  Column pass (ROWS false): the groups are the
// limb's columns (stride 2^n2); row pass: its contiguous blocks of 2^n2.  The
// first pass of a transform (FWD columns, inverse rows) converts the input to
// the working form, the second one gives canonical residues.
template <int LOGN, bool FWD, bool ROWS, int LPB, class BF, class LW, class V>
__device__ __forceinline__ void pass_body(const NttTabs& tb, const V (&v)[LPB], const bool (&live)[LPB], int w,
                                          LW* lds) {
    constexpr int n1 = LOGN / 2, n2 = LOGN - n1, LOGR = ROWS ? n2 : n1;
    constexpr int G = pass_groups(LOGR, LOGN - LOGR);
    using Gr = Grp<LOGR>;
    const int g = ROWS ? threadIdx.x / Gr::TG : threadIdx.x % G;
    const int t = ROWS ? threadIdx.x % Gr::TG : threadIdx.x / G;
    const int grp = w * G + g;
    auto at = [grp, t](int j) {
        return ROWS ? (grp << n2) + t + Gr::TG * j : ((t + Gr::TG * j) << n2) + grp;
    };
    constexpr bool FIRST = FWD != ROWS;
    constexpr bool FP = std::is_same_v<BF, BfFp>;
    constexpr bool PRE = HasPre<V>::value;
    constexpr bool LOAD_FP = FP && FIRST && HasLoadFp<V>::value;
    constexpr bool STORE_FP = FP && FWD && !FIRST && HasStoreFp<V>::value;
    u64 x[LPB][E], pre[LPB][PRE ? E : 1];
    BF kq[LPB];
    const u64* W[LPB];
    const u64* WS[LPB];
#pragma unroll
    for (int i = 0; i < LPB; ++i) {
        kq[i] = BF::of(tb.bc[v[i].basis]);
        if constexpr (HasBlock<V>::value) {
            v[i].load_block(kq[i], at, x[i]);
        } else if (live[i]) {
#pragma unroll
            for (int j = 0; j < E; ++j) {
                if constexpr (LOAD_FP) x[i][j] = BfFp::u(v[i].load_fp(at(j)));
                else x[i][j] = FIRST ? kq[i].in(v[i].load(at(j))) : v[i].load(at(j));
            }
            if constexpr (PRE) {
#pragma unroll
                for (int j = 0; j < E; ++j) pre[i][j] = v[i].pre(at(j));
            }
        }
        W[i] = (FWD ? tb.fwd : tb.inv) + (long long)v[i].basis * tb.N;
        WS[i] = (FWD ? tb.fwd_shoup : tb.inv_shoup) + (long long)v[i].basis * tb.N;
    }
    LW* my = lds + g * Gr::LDS;
    if constexpr (FWD) {
        if constexpr (ROWS)
            group_fwd_n<LOGR, LPB>(x, t, my, kq, W, WS,
                                   [grp](int s, int i) { return (1 << (n1 + s)) + (grp << s) + i; });
        else
            group_fwd_n<LOGR, LPB>(x, t, my, kq, W, WS, [](int s, int i) { return (1 << s) + i; });
    } else {
        if constexpr (ROWS)
            group_inv_n<LOGR, true, LPB>(x, t, my, kq, W, WS, [grp](int u, int i) {
                return (1 << (LOGN - 1 - u)) + (grp << (n2 - 1 - u)) + i;
            });
        else
            group_inv_n<LOGR, false, LPB>(x, t, my, kq, W, WS, [](int u, int i) { return (1 << (n1 - 1 - u)) + i; });
    }
#pragma unroll
    for (int i = 0; i < LPB; ++i) {
        if (!live[i]) continue;
        if constexpr (STORE_FP) {
#pragma unroll
            for (int j = 0; j < E; ++j) v[i].store_fp(at(j), BfFp::d(x[i][j]), PRE ? pre[i][PRE ? j : 0] : 0);
            continue;
        }
        if constexpr (!FIRST && FWD) {
#pragma unroll
            for (int j = 0; j < E; ++j) x[i][j] = kq[i].out_fwd(x[i][j]);
        }
        if constexpr (!FIRST && !FWD) {
            const u64* k = tb.bc[v[i].basis].inv_last;
            if constexpr (HasInvScale<V>::value) k = v[i].inv_scale;
#pragma unroll
            for (int j = 0; j < E / 2; ++j) kq[i].inv_last(x[i][j], x[i][j + E / 2], k);
        }
#pragma unroll
        for (int j = 0; j < E; ++j) {
            if constexpr (PRE) v[i].store_pre(at(j), x[i][j], pre[i][j]);
            else v[i].store(at(j), x[i][j]);
        }
    }
}

// The arithmetics a kernel holds.  With both, the compiler shares address
// registers across them and a pass takes up to 134 registers where either
// alone takes 100 to 106 (the integer forward column pass loses a wave per
// SIMD), so in-place batches whose moduli are of one kind get a kernel of their own.
enum class Arith { Both, Int, Fp };

// A workgroup's limbs (limb_views) through one pass in the arithmetic of their
// moduli; two limbs are interleaved only if both are integer limbs.
template <int LOGN, bool FWD, bool ROWS, int LPB, bool HALF, Arith A, class Job>
__device__ __forceinline__ void ntt_pass(const NttTabs& tb, const Job& job, int count) {
    constexpr int n1 = LOGN / 2, n2 = LOGN - n1;
    constexpr int wpl = ROWS ? pass_wpl(n2, n1) : pass_wpl(n1, n2);
    using LW = std::conditional_t<HALF, u32, u64>;  // LDS exchange word
    __shared__ LW lds[NTT_LDS_WORDS];
    using V = decltype(job.view(0));
    const int blk = blockIdx.x / wpl, w = blockIdx.x - blk * wpl;
    V v[LPB];
    bool live[LPB];
    if (!limb_views<LPB>(job, blk * LPB, count, v, live)) return;
    int fp = 0;
#pragma unroll
    for (int i = 0; i < LPB; ++i) fp += tb.fp(v[i].basis) ? 1 : 0;
    if constexpr (A == Arith::Int) {
        pass_body<LOGN, FWD, ROWS, LPB, BfInt>(tb, v, live, w, lds);
    } else if constexpr (A == Arith::Fp) {
        pass_body<LOGN, FWD, ROWS, LPB, BfFp>(tb, v, live, w, lds);
    } else if constexpr (LPB == 1) {
        if (fp) pass_body<LOGN, FWD, ROWS, 1, BfFp>(tb, v, live, w, lds);
        else pass_body<LOGN, FWD, ROWS, 1, BfInt>(tb, v, live, w, lds);
    } else if (fp == 0) {
        pass_body<LOGN, FWD, ROWS, LPB, BfInt>(tb, v, live, w, lds);
    } else {
        static_assert(LPB == 2, "one or two limbs per workgroup");
        const bool l1[1] = {true};
#pragma unroll 1
        for (int i = 0; i < 2; ++i) {
            if (!(i ? live[1] : live[0])) continue;  // uniform
            const V v1[1] = {i ? v[1] : v[0]};
            __syncthreads();  // the previous limb's LDS reads are done
            if (tb.fp(v1[0].basis)) pass_body<LOGN, FWD, ROWS, 1, BfFp>(tb, v1, l1, w, lds);
            else pass_body<LOGN, FWD, ROWS, 1, BfInt>(tb, v1, l1, w, lds);
        }
    }
}

template <int LOGN, bool FWD, int LPB, bool HALF, Arith A, class Job>
__global__ void __launch_bounds__(NTT_THREADS) k_ntt_cols(NttTabs tb, Job job, int count) {
    ntt_pass<LOGN, FWD, false, LPB, HALF, A>(tb, job, count);
}
template <int LOGN, bool FWD, int LPB, bool HALF, Arith A, class Job>
__global__ void __launch_bounds__(NTT_THREADS) k_ntt_rows(NttTabs tb, Job job, int count) {
    ntt_pass<LOGN, FWD, true, LPB, HALF, A>(tb, job, count);
}
// The same pass held to 128 VGPRs (four waves per SIMD, the LDS limit), for
// jobs whose load or store does enough work of its own that the scheduler
// would otherwise trade occupancy for loads hoisted across the whole pass.
template <int LOGN, bool FWD, Arith A, class Job>
__global__ void __launch_bounds__(NTT_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
k_ntt_rows_w4(NttTabs tb, Job job, int count) {
    ntt_pass<LOGN, FWD, true, 1, false, A>(tb, job, count);
}

#define MI_NTT_LOGN_CASES(K)                                                                          \
    switch (c.logN) {                                                                                 \
        case 10: K(10); break;                                                                        \
        case 11: K(11); break;                                                                        \
        case 12: K(12); break;                                                                        \
        case 13: K(13); break;                                                                        \
        case 14: K(14); break;                                                                        \
        case 15: K(15); break;                                                                        \
        case 16: K(16); break;                                                                        \
        default: throw Error(-1, "ntt: unsupported ring dimension");                                  \
    }

template <bool FWD, int LPB, bool HALF, Arith A = Arith::Both, class Job>
void launch_cols(const Context& c, const Job& job, int count, hipStream_t s) {
    if (count >= (1 << 20)) throw Error(-1, "ntt: more than 2^20 limbs in one launch");
    const NttTabs tb = tabs_of(c);
    const unsigned blocks = (unsigned)((count + LPB - 1) / LPB);
#define MI_COLS(LN)                                                                                   \
    hipLaunchKernelGGL((k_ntt_cols<LN, FWD, LPB, HALF, A, Job>), dim3(blocks * pass_wpl(LN / 2, LN - LN / 2)), \
                       dim3(pass_threads(LN / 2, LN - LN / 2)), 0, s, tb, job, count)
    MI_NTT_LOGN_CASES(MI_COLS)
#undef MI_COLS
    MI_HIP(hipGetLastError());
}

template <bool FWD, int LPB, bool HALF, Arith A = Arith::Both, class Job>
void launch_rows(const Context& c, const Job& job, int count, hipStream_t s) {
    if (count >= (1 << 20)) throw Error(-1, "ntt: more than 2^20 limbs in one launch");
    const NttTabs tb = tabs_of(c);
    const unsigned blocks = (unsigned)((count + LPB - 1) / LPB);
#define MI_ROWS(LN)                                                                                   \
    hipLaunchKernelGGL((k_ntt_rows<LN, FWD, LPB, HALF, A, Job>), dim3(blocks * pass_wpl(LN - LN / 2, LN / 2)), \
                       dim3(pass_threads(LN - LN / 2, LN / 2)), 0, s, tb, job, count)
    MI_NTT_LOGN_CASES(MI_ROWS)
#undef MI_ROWS
    MI_HIP(hipGetLastError());
}

template <bool FWD, Arith A = Arith::Both, class Job>
void launch_rows_w4(const Context& c, const Job& job, int count, hipStream_t s) {
    if (count >= (1 << 20)) throw Error(-1, "ntt: more than 2^20 limbs in one launch");
    const NttTabs tb = tabs_of(c);
#define MI_ROWS(LN)                                                                                   \
    hipLaunchKernelGGL((k_ntt_rows_w4<LN, FWD, A, Job>), dim3((unsigned)count * pass_wpl(LN - LN / 2, LN / 2)), \
                       dim3(pass_threads(LN - LN / 2, LN / 2)), 0, s, tb, job, count)
    MI_NTT_LOGN_CASES(MI_ROWS)
#undef MI_ROWS
    MI_HIP(hipGetLastError());
}

// One pass of an in-place batch (mi_ntt.hip) in configuration `variant` of the
// NTT plan: 1 = one limb per workgroup, 2 = two limbs per workgroup, 3 = one
// limb with the LDS exchanges in 32-bit halves.
void launch_plain_pass(const Context& c, bool fwd, bool rows, int variant, const PlainJob& job, int count,
                       hipStream_t s);

// One pass of a transform: in-place batches in the configuration the
// context's tuned plan gives for the launch size, the fused jobs with one
// limb per workgroup.  Contexts of integers alone take that arithmetic's kernel:
// over 60-bit limbs, integer kernels only / kernels that hold both / now, us,
// rescale of two polys of 8 limbs at N = 2^14 31.6 / 32.2 / 31.6, ModDown of one
// of 12 + 4 at N = 2^15 36.1 / 36.7 / 35.9.
template <bool FWD, bool ROWS, class Job>
void launch_pass(const Context& c, const Job& job, int count, hipStream_t s) {
    if constexpr (std::is_same_v<Job, PlainJob>) {
        launch_plain_pass(c, FWD, ROWS, c.ntt_variant(count), job, count, s);
    } else if (c.integer_only()) {
        if constexpr (ROWS) launch_rows<FWD, 1, false, Arith::Int>(c, job, count, s);
        else launch_cols<FWD, 1, false, Arith::Int>(c, job, count, s);
    } else {
        if constexpr (ROWS) launch_rows<FWD, 1, false>(c, job, count, s);
        else launch_cols<FWD, 1, false>(c, job, count, s);
    }
}

// Forward NTT: first pass runs job `in` (load input, store intermediate),
// second pass runs job `out` (load intermediate, store output).
template <class JobIn, class JobOut>
void run_ntt_fwd(const Context& c, const JobIn& in, const JobOut& out, int count, hipStream_t s) {
    const long probe = c.probe_open(s, count);
    launch_pass<true, false>(c, in, count, s);
    launch_pass<true, true>(c, out, count, s);
    c.probe_close(probe, s);
}
template <class JobIn, class JobOut>
void run_ntt_inv(const Context& c, const JobIn& in, const JobOut& out, int count, hipStream_t s) {
    const long probe = c.probe_open(s, count);
    launch_pass<false, true>(c, in, count, s);
    launch_pass<false, false>(c, out, count, s);
    c.probe_close(probe, s);
}

// Evaluation-domain source index of output index i under Galois element g:
// dst[brev(d)] = src[brev(((2d+1) g mod 2N - 1) / 2)].
__device__ __forceinline__ u32 galois_index(u32 i, u64 g, int logN) {
    const u32 mask2n = (2u << logN) - 1;
    const u32 d = __brev(i) >> (32 - logN);
    const u32 e = (u32)(((u64)(2 * d + 1) * g) & mask2n);
    return __brev((e - 1) >> 1) >> (32 - logN);
}

// Block -> (item, slot, tile) with the blocks of one (slot, tile) for all
// items consecutive on one XCD: workgroups are dealt to the 8 XCDs round
// robin, so block b runs on XCD b % 8.  The key (or diagonal) tile that all
// items read is then fetched once into that XCD's L2.
struct TileMap {
    int item, slot, tile;
    bool valid;
};
__device__ __forceinline__ TileMap map_tile(int b, int items, int tiles_per_slot, int slots) {
    const int xcd = b & 7, local = b >> 3;
    const int it = local % items, tl = local / items;
    const int tile = tl * 8 + xcd;
    TileMap m;
    m.item = it;
    m.slot = tile / tiles_per_slot;
    m.tile = tile - m.slot * tiles_per_slot;
    m.valid = m.slot < slots;
    return m;
}
inline unsigned tile_grid(int items, int tiles_per_slot, int slots) {
    const long long tiles = (long long)tiles_per_slot * slots;
    return (unsigned)(((tiles + 7) / 8) * 8 * items);
}

}  // namespace mi
