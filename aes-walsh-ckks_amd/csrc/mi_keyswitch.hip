// Hybrid key switching (reference ckks_hybrid_key_switch_inplace,
// ckks_keyswitch.cpp:1330-1641, fold_hybrid_keyswitch = true), hoisting
// (ckks_hoist_ciphertext_a_qp_eval, :344-373) and the QP-basis variants
// (:675-1328).
//
// Steps, each a device routine reused by the linear transform:
//   ks_modup     C = INTT(key term); D[d] = HPS ModUp of digit d's limbs of C
//                to the other Q limbs and P, the digit's own limbs copied from
//                the evaluation-domain key term (:278-332, :1452); NTT of D.
//   k_mac        acc = sum_d D[d] * key[d] per QP slot (Montgomery REDC or
//                Barrett), written either split (Q slots combined into the
//                outputs with Add/Assign, P slots kept for ModDown) or whole in
//                the QP basis, optionally through a Galois automorphism and
//                with a b term added (:675-852, :373-416).
//   ks_moddown   folded ModDown (:521-673, mi_moddown.hip), also with the key
//                inner product folded in (mi_moddown_mac.hpp).
// Reordering "+ acc" before "- NTT(contribution)" leaves every canonical
// residue unchanged.
#include "mi_extend.hpp"
#include "mi_moddown.hpp"

#include <algorithm>
#include <vector>

namespace mi {

// ---- inverse NTT of n key terms -> C (item-minor within a limb) ----
// The first pass also copies each limb, as it is read, to its own place among
// the digits: all words loaded before the first is stored (a later load may
// not pass a store that it might overlap, and each would wait for its own).
struct CopyListJob {
    const u64* src[KS_MAX_ITEMS];
    u64* dst;
    long long dstride;
    u64* digits;  // item i's [parts][L+K][N] at digits + i * digit_stride
    long long digit_stride;
    int n, alpha, slots;
    u64 N;
    FastDiv per_limb, per_digit;  // n, alpha
    struct View {
        int basis;
        const u64* s;
        u64* d;
        u64* own;
        static constexpr bool BLOCK = true;
        template <class BF, class AT>
        __device__ __forceinline__ void load_block(const BF& bf, AT at, u64 (&x)[E]) const {
#pragma unroll
            for (int j = 0; j < E; ++j) x[j] = s[at(j)];
#pragma unroll
            for (int j = 0; j < E; ++j) {
                own[at(j)] = x[j];
                x[j] = bf.in(x[j]);
            }
        }
        __device__ void store(int i, u64 v) const { d[i] = v; }
    };
    __device__ View view(int k) const {
        const int l = per_limb.div(k), it = k - l * n;
        const long long o = (long long)l * N;
        return View{l, src[it] + o, dst + it * dstride + o,
                    digits + it * digit_stride + (long long)per_digit.div(l) * slots * N + o};
    }
    __device__ bool skip(int) const { return false; }
};
// Second pass: C holds y = x qhat^-1 mod q of the limb's digit, a factor that
// rides in the last stage's N^-1.
struct ScaledListJob {
    u64* dst;
    long long dstride;
    int n, alpha;
    const u64* inv_scale[16];  // per digit [ns][4]
    u64 N;
    FastDiv per_limb, per_digit;
    struct View {
        int basis;
        u64* p;
        const u64* inv_scale;
        __device__ u64 load(int i) const { return p[i]; }
        __device__ void store(int i, u64 v) const { p[i] = v; }
    };
    __device__ View view(int k) const {
        const int l = per_limb.div(k), it = k - l * n, d = per_digit.div(l);
        return View{l, dst + it * dstride + (long long)l * N, inv_scale[d] + 4 * (l - d * alpha)};
    }
    __device__ bool skip(int) const { return false; }
};

// ---- ModUp of all digits of n items, fused with the forward column pass ----
struct ModUpJob {
    ExtGrid grid;
    const u64* coeff;  // C: item i's [L][N] at coeff + i*L*N
    u64* digits;       // item i's D [parts][L+K][N] at digits + i*dstride
    long long dstride;
    int L, K, nq, parts;
    u64 N;
    FastDiv per_item;  // parts
    int s0[16];
    ExtTables t[16];
    const BasisConst* bc;
    // source: item-major (item, digit)
    __device__ int targets(int source) const { return t[source - per_item.div(source) * parts].nd; }
    __device__ ExtView view(int source, int target) const {
        const int it = per_item.div(source), d = source - it * parts;
        const ExtTables& e = t[d];
        // targets in order: chain limbs before the digit, after it, P limbs
        const int slot = target < s0[d] ? target : target + e.ns;
        const int basis = slot < L ? slot : nq + (slot - L);
        const BasisConst b = bc[basis];
        return ExtView{basis,
                       coeff + ((long long)it * L + s0[d]) * N,
                       digits + it * dstride + ((long long)d * (L + K) + slot) * N,
                       (long long)N,
                       e.terms + (long long)target * e.ns,
                       e.src_inv,
                       e.corr + 2 * target,
                       e.ns,
                       e.wide,
                       b.qninv,
                       b.mu_hi};
    }
};

// ---- forward NTT of the ModUp'd slots ----
struct DigitJob {
    u64* digits;
    long long dstride;
    int L, K, nq, alpha, parts, n;
    u64 N;
    FastDiv per_slot, per_item;  // parts * n, parts
    struct View {
        int basis;
        u64* p;
        __device__ u64 load(int i) const { return p[i]; }
        __device__ void store(int i, u64 v) const { p[i] = v; }
    };
    // slot-major: every item's and digit's slot 0, then slot 1, ... (shared twiddles)
    __device__ void split(int k, int& l, int& it, int& d) const {
        l = per_slot.div(k);
        const int r = k - l * (parts * n);
        it = per_item.div(r);
        d = r - it * parts;
    }
    __device__ View view(int k) const {
        int l, it, d;
        split(k, l, it, d);
        return View{l < L ? l : nq + (l - L), digits + it * dstride + ((long long)d * (L + K) + l) * N};
    }
    __device__ bool skip(int k) const {
        int l, it, d;
        split(k, l, it, d);
        const int s0 = d * alpha;
        return l >= s0 && l < s0 + alpha && l < L;
    }
};

void ks_modup_n(Context& c, int level, int n, const u64* const* key_terms, u64* D, long long dstride,
                u64* C, hipStream_t s) {
    const int L = level + 1, K = c.np, parts = c.parts(level);
    const u64 N = c.N;
    if (n < 1 || n > KS_MAX_ITEMS) throw Error(-1, "ModUp batch size out of range");
    if (parts > 16) throw Error(-1, "too many digits");
    for (int d = 0; d < parts; ++d)
        if (c.modup[level][d].ext.ns > MAX_ALPHA) throw Error(-1, "digit wider than 16 limbs");
    {
        CopyListJob in{};
        ScaledListJob out{};
        for (int i = 0; i < n; ++i) in.src[i] = key_terms[i];
        for (int d = 0; d < parts; ++d) out.inv_scale[d] = c.modup[level][d].inv_scale;
        in.dst = out.dst = C;
        in.dstride = out.dstride = (long long)L * (long long)N;
        in.digits = D;
        in.digit_stride = dstride;
        in.slots = L + K;
        in.n = out.n = n;
        in.alpha = out.alpha = c.alpha;
        in.N = out.N = N;
        in.per_limb = out.per_limb = fast_div(n);
        in.per_digit = out.per_digit = fast_div(c.alpha);
        run_ntt_inv(c, in, out, L * n, s);
    }
    ModUpJob m{};
    m.coeff = C;
    m.digits = D;
    m.dstride = dstride;
    m.L = L;
    m.K = K;
    m.nq = c.nq;
    m.parts = parts;
    m.N = N;
    m.per_item = fast_div(parts);
    m.bc = c.d_bc;
    int maxnd = 1;
    for (int d = 0; d < parts; ++d) {
        m.s0[d] = c.modup[level][d].s0;
        m.t[d] = c.modup[level][d].ext;
        maxnd = std::max(maxnd, m.t[d].nd);
    }
    const DigitJob j{D, dstride, L, K, c.nq, c.alpha, parts, n, N, fast_div(parts * n), fast_div(parts)};
    const int limbs = parts * (L + K) * n;
    const long probe = c.probe_open(s, limbs);
    launch_ext_cols(c, m, n * parts, maxnd, s);
    launch_pass<true, true>(c, j, limbs, s);
    c.probe_close(probe, s);
}

void ks_modup(Context& c, int level, const u64* key_term, u64* D, u64* C, hipStream_t s) {
    const u64* kt[1] = {key_term};
    ks_modup_n(c, level, 1, kt, D, 0, C, s);
}

// ---- key inner product ----
__global__ void __launch_bounds__(KS_THREADS) k_mac(MacArgs a) {
    const u64 N = (u64)1 << a.logN;
    const int slots = a.L + a.K;
    const int tps = (int)(N / KS_THREADS);
    const TileMap m = map_tile(blockIdx.x, a.items, tps, slots);
    if (!m.valid) return;
    const int it = m.item, slot = m.slot;
    const long long i = (long long)m.tile * KS_THREADS + threadIdx.x;
    const int basis = slot < a.L ? slot : a.nq + (slot - a.L);
    const int key_limbs = a.nq + a.K;
    const BasisConst b = a.bc[basis];
    const long long src = a.galois ? (long long)galois_index((u32)i, a.galois, a.logN) : i;
    const u64* digits = a.digits + it * a.digits_stride;
    const u64* key = a.key[it];
    u64 acc_b, acc_a;
    const u64* dg = digits + (long long)slot * N + src;
    const u64* kp = key + (long long)basis * N + src;
    const long long dstep = (long long)slots * N, kstep = 2LL * key_limbs * N, to_a = (long long)key_limbs * N;
    // Operands are residues below 4q.
    if (b.fp) {  // uniform over the block
        // each product at most 13/2 q (FpMod::mulq), centred; 16 of them stay at 8q
        const FpMod m{b.qd, b.inv_d};
        double sb = 0.0, sa = 0.0;
        for (int d = 0; d < a.parts; ++d) {
            const double x = fp_from_u64(dg[d * dstep]);
            const u64* k = kp + d * kstep;
            sb += m.centred(m.mulq(x, fp_from_u64(k[0])));
            sa += m.centred(m.mulq(x, fp_from_u64(k[to_a])));
        }
        if (a.montgomery) {
            sb = m.mul(sb, b.rinv_fp, b.rinv_fpq);
            sa = m.mul(sa, b.rinv_fp, b.rinv_fpq);
        }
        acc_b = m.canonical(sb);
        acc_a = m.canonical(sa);
    } else {
        // Exact 128-bit sums.  Up to 3 products below 16 q^2 (q < 2^61) fit and
        // their high word is reduced once; otherwise the operands are brought
        // below q and at most 16 products of residues below 2^62 fit.  One
        // reduction at the end (REDC for Montgomery-form keys, Barrett
        // otherwise) gives the canonical residue of the sum.
        U128 sb{0, 0}, sa{0, 0};
        const bool lazy = a.parts <= 3 && b.q < (1ull << 61);
        for (int d = 0; d < a.parts; ++d) {
            const u64* k = kp + d * kstep;
            u64 x = dg[d * dstep], kbv = k[0], kav = k[to_a];
            if (!lazy) {
                x = reduce_4q(x, b.q);
                kbv = reduce_4q(kbv, b.q);
                kav = reduce_4q(kav, b.q);
            }
            mac128(sb, x, kbv);
            mac128(sa, x, kav);
        }
        sb.hi = reduce64(sb.hi, b.q, b.mu_hi);
        sa.hi = reduce64(sa.hi, b.q, b.mu_hi);
        if (a.montgomery) {
            acc_b = redc128(sb.lo, sb.hi, b.q, b.qninv);
            acc_a = redc128(sa.lo, sa.hi, b.q, b.qninv);
        } else {
            acc_b = barrett128(sb.lo, sb.hi, b.q, b.mu_lo, b.mu_hi);
            acc_a = barrett128(sa.lo, sa.hi, b.q, b.mu_lo, b.mu_hi);
        }
    }
    const u64* ib = a.init_b[it];
    if (ib && slot < a.L) acc_b = add_mod(acc_b, ib[(long long)slot * N + src], b.q);
    if (a.qp_out) {
        const u64* ab = a.add_b[it];
        if (ab) acc_b = add_mod(acc_b, ab[(long long)slot * N + src], b.q);
        u64* pb = a.b_out[it] + (long long)slot * N + i;
        u64* pa = a.a_out[it] + (long long)slot * N + i;
        *pb = a.accumulate ? add_mod(*pb, acc_b, b.q) : acc_b;
        *pa = a.accumulate ? add_mod(*pa, acc_a, b.q) : acc_a;
    } else if (slot < a.L) {
        u64* pb = a.b_out[it] + (long long)slot * N + i;
        u64* pa = a.a_out[it] + (long long)slot * N + i;
        *pb = a.b_mode == 0 ? add_mod(*pb, acc_b, b.q) : acc_b;
        *pa = a.a_mode == 0 ? add_mod(*pa, acc_a, b.q) : acc_a;
    } else {
        const int pi = slot - a.L;
        u64* ap = a.accp + it * a.accp_stride;
        ap[(long long)pi * N + i] = acc_a;
        ap[((long long)a.K + pi) * N + i] = acc_b;
    }
}

void ks_mac(const Context& c, const MacArgs& args, int level, hipStream_t s) {
    if (args.items < 1 || args.items > KS_MAX_ITEMS) throw Error(-1, "key product batch size out of range");
    if (args.parts < 1 || args.parts > 16) throw Error(-1, "too many digits");  // 128-bit sums hold 16 products
    const int tps = (int)(c.N / KS_THREADS);
    const unsigned blocks = tile_grid(args.items, tps, level + 1 + c.np);
    hipLaunchKernelGGL(k_mac, dim3(blocks), dim3(KS_THREADS), 0, s, args);
    MI_HIP(hipGetLastError());
}

MacArgs mac_args(const Context& c, int level, const u64* digits, const u64* key, bool montgomery) {
    MacArgs a{};
    a.digits = digits;
    a.key[0] = key;
    a.items = 1;
    a.L = level + 1;
    a.K = c.np;
    a.nq = c.nq;
    a.parts = c.parts(level);
    a.logN = c.logN;
    a.montgomery = montgomery ? 1 : 0;
    a.bc = c.d_bc;
    return a;
}

// ---------------------------------------------------------------- entry points
size_t ks_item_words(const Context& c, int level) {
    const size_t L = level + 1, K = c.np, parts = c.parts(level), N = c.N;
    return (L + parts * (L + K) + 2 * K + 2 * L) * N;
}

void keyswitch_items(Context& c, const KsItem* items, int n, bool montgomery, hipStream_t s) {
    if (n < 1 || n > KS_MAX_ITEMS) throw Error(-1, "key switch batch size out of range");
    // A single switch (a relinearisation, say) sizes the workspace for a rotation
    // at its level too: growing it later would stop the stream for a new allocation.
    const size_t staging = n == 1 ? 2 * (size_t)(items[0].level + 1) * c.N : 0;
    const size_t need = sizeof(u64) * ks_item_words(c, items[0].level) * (size_t)n;
    bool whole;
    u64* ws = (u64*)c.workspace_up_to(s, need + sizeof(u64) * staging, need, &whole);
    keyswitch_items_with(c, items, n, montgomery, ws, s);
}

void keyswitch_items_with(Context& c, const KsItem* items, int n, bool montgomery, u64* ws, hipStream_t s) {
    if (n < 1 || n > KS_MAX_ITEMS) throw Error(-1, "key switch batch size out of range");
    const int level = items[0].level;
    for (int i = 1; i < n; ++i)
        if (items[i].level != level || items[i].b_mode != items[0].b_mode || items[i].a_mode != items[0].a_mode)
            throw Error(-1, "key switch batch items must share level and combine modes");
    const int L = level + 1, K = c.np, parts = c.parts(level);
    const u64 N = c.N;
    const long long dw = (long long)parts * (L + K) * (long long)N;
    u64* C = ws;
    u64* D = C + (size_t)n * L * N;
    u64* AP = D + (size_t)n * dw;
    u64* T = AP + (size_t)n * 2 * K * N;
    const u64* kt[KS_MAX_ITEMS];
    for (int i = 0; i < n; ++i) kt[i] = items[i].key_term;
    ks_modup_n(c, level, n, kt, D, dw, C, s);
    if (parts <= 3 && c.fuse_mac) {
        ks_moddown_mac(c, level, n, items, D, dw, AP, T, montgomery, s);
        return;
    }
    MacArgs a = mac_args(c, level, D, items[0].key, montgomery);
    a.items = n;
    a.digits_stride = dw;
    a.accp = AP;
    a.accp_stride = 2LL * K * (long long)N;
    a.b_mode = items[0].b_mode;
    a.a_mode = items[0].a_mode;
    for (int i = 0; i < n; ++i) {
        a.key[i] = items[i].key;
        a.b_out[i] = items[i].b_out;
        a.a_out[i] = items[i].a_out;
        a.init_b[i] = items[i].init_b;
    }
    ks_mac(c, a, level, s);
    u64* p[2 * KS_MAX_ITEMS];
    const u64* base[2 * KS_MAX_ITEMS];
    u64* out[2 * KS_MAX_ITEMS];
    for (int i = 0; i < n; ++i) {
        p[2 * i] = AP + (size_t)i * 2 * K * N;
        p[2 * i + 1] = p[2 * i] + (size_t)K * N;
        base[2 * i] = out[2 * i] = items[i].a_out;
        base[2 * i + 1] = out[2 * i + 1] = items[i].b_out;
    }
    ks_moddown_n(c, level, 2 * n, p, base, out, T, s);
}

void keyswitch(Context& c, const KsItem& it, bool montgomery, hipStream_t s) {
    if (it.level < 0 || it.level >= c.nq) throw Error(-1, "invalid ciphertext level");
    keyswitch_items(c, &it, 1, montgomery, s);
}

namespace {
struct Span {
    const u64* lo;
    const u64* hi;
};
bool overlaps(const Span& x, const Span& y) { return x.lo < y.hi && y.lo < x.hi; }
}  // namespace

// Groups of one (level, modes) whose buffers are independent, up to the
// tuned group size (at most KS_MAX_ITEMS) each.  An item that touches a buffer an earlier item of the
// open group of its kind writes (or writes one it reads) closes that group
// and every other open group, so the order of dependent switches is kept.
void keyswitch_batch(Context& c, const KsItem* items, int n, bool montgomery, hipStream_t s) {
    struct Group {
        int level, b_mode, a_mode;
        std::vector<KsItem> v;
        std::vector<Span> writes, reads;
        bool full = false;
    };
    std::vector<Group> open;
    // Open groups (full ones included) are independent of each other: they
    // run spread over the caller's stream and the side streams, forked from
    // it and joined back, so groups overlap each other's fill and drain.
    auto flush_all = [&]() {
        std::vector<const Group*> gs;
        for (const auto& g : open)
            if (!g.v.empty()) gs.push_back(&g);
        if (gs.size() == 1 || (!gs.empty() && !c.multi_stream)) {
            for (const Group* g : gs) keyswitch_items(c, g->v.data(), (int)g->v.size(), montgomery, s);
        } else if (gs.size() > 1) {
            const auto& side = c.side_streams();
            const size_t ns = std::min(gs.size(), side.size() + 1);
            hipEvent_t fork;
            MI_HIP(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
            MI_HIP(hipEventRecord(fork, s));
            for (size_t k = 1; k < ns; ++k) MI_HIP(hipStreamWaitEvent(side[k - 1], fork, 0));
            for (size_t g = 0; g < gs.size(); ++g) {
                hipStream_t st = g % ns == 0 ? s : side[g % ns - 1];
                keyswitch_items(c, gs[g]->v.data(), (int)gs[g]->v.size(), montgomery, st);
            }
            for (size_t k = 1; k < ns; ++k) {
                hipEvent_t j;
                MI_HIP(hipEventCreateWithFlags(&j, hipEventDisableTiming));
                MI_HIP(hipEventRecord(j, side[k - 1]));
                MI_HIP(hipStreamWaitEvent(s, j, 0));
                MI_HIP(hipEventDestroy(j));
            }
            MI_HIP(hipEventDestroy(fork));
        }
        open.clear();
    };
    for (int i = 0; i < n; ++i) {
        const KsItem& it = items[i];
        const size_t W = (size_t)(it.level + 1) * c.N;
        const Span rd{it.key_term, it.key_term + W};
        const Span ri{it.init_b, it.init_b ? it.init_b + W : it.init_b};
        const Span wb{it.b_out, it.b_out + W}, wa{it.a_out, it.a_out + W};
        bool conflict = false;
        for (const auto& g : open) {
            for (const auto& w : g.writes)
                if (overlaps(w, rd) || overlaps(w, ri) || overlaps(w, wb) || overlaps(w, wa)) conflict = true;
            for (const auto& r : g.reads)
                if (overlaps(r, wb) || overlaps(r, wa)) conflict = true;
        }
        if (conflict) flush_all();
        Group* g = nullptr;
        for (auto& x : open)
            if (!x.full && x.level == it.level && x.b_mode == it.b_mode && x.a_mode == it.a_mode) g = &x;
        if (!g) {
            open.push_back(Group{it.level, it.b_mode, it.a_mode, {}, {}, {}, false});
            g = &open.back();
        }
        g->v.push_back(it);
        g->writes.push_back(wb);
        g->writes.push_back(wa);
        g->reads.push_back(rd);
        if (it.init_b) g->reads.push_back(Span{it.init_b, it.init_b + W});
        if ((int)g->v.size() == c.tune.ks_group) g->full = true;  // runs at the next flush, with the others
    }
    flush_all();
}

void hoist(Context& c, int level, const u64* a_eval, u64* digits, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    u64* C = (u64*)c.workspace(s, sizeof(u64) * (size_t)(level + 1) * c.N);
    ks_modup(c, level, a_eval, digits, C, s);
}

void hoist_batch(Context& c, int level, int n, const u64* const* a_eval, u64* digits, long long dstride,
                 hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    if (n < 1) throw Error(-1, "need at least one ciphertext");
    for (int i0 = 0; i0 < n; i0 += KS_MAX_ITEMS) {
        const int m = std::min(KS_MAX_ITEMS, n - i0);
        u64* C = (u64*)c.workspace(s, sizeof(u64) * (size_t)m * (level + 1) * c.N);
        ks_modup_n(c, level, m, a_eval + i0, digits + (long long)i0 * dstride, dstride, C, s);
    }
}

void keyswitch_hoisted(Context& c, int level, const u64* digits, const u64* key, u64* b_out,
                       u64* a_out, int b_mode, int a_mode, u64 galois, bool montgomery, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    const int L = level + 1, K = c.np;
    const u64 N = c.N;
    const size_t words = (size_t)(2 * K + 2 * L + (galois ? 2 * L : 0)) * N;
    u64* AP = (u64*)c.workspace(s, sizeof(u64) * words);
    u64* T = AP + (size_t)2 * K * N;
    MacArgs a = mac_args(c, level, digits, key, montgomery);
    a.b_out[0] = b_out;
    a.a_out[0] = a_out;
    a.b_mode = b_mode;
    a.a_mode = a_mode;
    a.accp = AP;
    ks_mac(c, a, level, s);
    ks_moddown(c, level, AP, AP + (size_t)K * N, a_out, b_out, a_out, b_out, T, s);
    if (galois) {
        u64* tmp = T + (size_t)2 * L * N;
        const long long W = (long long)L * (long long)N;
        automorphism(c, L, galois, b_out, tmp, 1, W, W, s);
        automorphism(c, L, galois, a_out, tmp + W, 1, W, W, s);
        MI_HIP(hipMemcpyAsync(b_out, tmp, sizeof(u64) * W, hipMemcpyDeviceToDevice, s));
        MI_HIP(hipMemcpyAsync(a_out, tmp + W, sizeof(u64) * W, hipMemcpyDeviceToDevice, s));
    }
}

// dst_a[i], dst_b[i] = automorphism g_i of item i's (a, b) pair at src + i*2*L*N
struct AutoItemsArgs {
    const u64* src;
    u64 galois[KS_MAX_ITEMS];
    u64* dst_a[KS_MAX_ITEMS];
    u64* dst_b[KS_MAX_ITEMS];
    int L, logN;
};

__global__ void __launch_bounds__(KS_THREADS) k_automorphism_items(AutoItemsArgs a) {
    const u64 N = (u64)1 << a.logN;
    const int tps = (int)(N / KS_THREADS);
    const int tile = blockIdx.x % tps, rest = blockIdx.x / tps;
    const int l = rest % a.L, poly = (rest / a.L) & 1, it = rest / (2 * a.L);
    const u32 i = (u32)tile * KS_THREADS + threadIdx.x;
    const u32 sidx = galois_index(i, a.galois[it], a.logN);
    const u64* src = a.src + ((long long)it * 2 + poly) * a.L * N + (long long)l * N;
    u64* dst = (poly == 0 ? a.dst_a[it] : a.dst_b[it]) + (long long)l * N;
    dst[i] = src[sidx];
}

// Whether an output pair of hoisted rotations overlaps the digits or a key.
static bool outputs_overlap_reads(const Context& c, int level, const u64* digits, long long dstride, int period, int n,
                                  const u64* const* keys, u64* const* b_out, u64* const* a_out) {
    const long long N = (long long)c.N, W = (level + 1) * N, parts = c.parts(level);
    const long long digit_words = (period - 1) * dstride + parts * (level + 1 + c.np) * N;
    const long long key_words = parts * 2 * c.nb() * N;
    std::vector<const u64*> ks(keys, keys + n);
    std::sort(ks.begin(), ks.end());
    ks.erase(std::unique(ks.begin(), ks.end()), ks.end());
    for (int i = 0; i < n; ++i)
        for (const u64* o : {(const u64*)b_out[i], (const u64*)a_out[i]}) {
            if (overlaps(Span{o, o + W}, Span{digits, digits + digit_words})) return true;
            const auto k = std::lower_bound(ks.begin(), ks.end(), o + W);  // the last key that starts below the output's end
            if (k != ks.begin() && *(k - 1) + key_words > o) return true;
        }
    return false;
}

void rotate_hoisted_items(Context& c, int level, const u64* digits, long long dstride, int period,
                          const u64* const* b, int n, const u64* galois, const u64* const* keys, u64* const* b_out,
                          u64* const* a_out, bool montgomery, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    if (n < 1) throw Error(-1, "need at least one rotation");
    if (period < 1 || period > n) period = n;
    const int L = level + 1, K = c.np;
    const u64 N = c.N;
    const long long LN = (long long)L * (long long)N, KN = (long long)K * (long long)N;
    // item i reads the hoist at digits + (i mod period) * dstride: chunks of
    // up to the group size inside each run of `period` items
    const int chunk = std::min(period, c.tune.ks_group);
    const int per_block = (period + chunk - 1) / chunk;
    const int nblocks = (n + period - 1) / period;
    const bool fold = c.parts(level) <= 3 && c.fuse_mac;
    // Folded, the last pass stores through the rotation's map while other
    // workgroups still read the digits and keys: outputs on their memory (an
    // output may take a buffer that the chunk no longer needs) go through staging.
    const bool mapped = fold && !outputs_overlap_reads(c, level, digits, dstride, period, n, keys, b_out, a_out);
    // per rotation: P accumulators (a, b) | ModDown temp | switched pair (a, b; not mapped)
    const size_t ws_bytes = sizeof(u64) * (size_t)chunk * (2 * KN + (mapped ? 2 : 4) * LN);
    over_streams(c, s, nblocks * per_block, ws_bytes, [&](hipStream_t st, u64* ws, int ci) {
        const int blk = ci / per_block, cb = ci - blk * per_block;
        const int i0 = blk * period + cb * chunk;
        if (i0 >= n) return;
        const int m = std::min(std::min(chunk, period - cb * chunk), n - i0);
        u64* AP = ws;
        u64* Tm = AP + chunk * 2 * KN;
        u64* SW = Tm + chunk * 2 * LN;
        const u64* dig = digits + (long long)(cb * chunk) * dstride;
        // key products of the hoisted digits, b added in the Q limbs
        // (ckks_hybrid_key_switch_hoisted_inplace with b Add, a Assign): mapped,
        // the last pass stores through the rotation's map; else into staging
        // pairs, permuted by a pass of their own
        if (fold) {
            KsItem items[KS_MAX_ITEMS];
            for (int it = 0; it < m; ++it) {
                items[it] = KsItem{nullptr, keys[i0 + it], b_out[i0 + it], a_out[i0 + it], level, 1, 1, b[i0 + it],
                                   galois[i0 + it] % (2 * N)};
                if (mapped) continue;
                items[it].a_out = SW + it * 2 * LN;
                items[it].b_out = SW + it * 2 * LN + LN;
                items[it].galois = 0;
            }
            ks_moddown_mac(c, level, m, items, dig, dstride, AP, Tm, montgomery, st);
            if (mapped) return;
        } else {
            MacArgs ma = mac_args(c, level, dig, keys[i0], montgomery);
            ma.items = m;
            ma.digits_stride = dstride;
            ma.accp = AP;
            ma.accp_stride = 2 * KN;
            ma.b_mode = 1;
            ma.a_mode = 1;
            for (int it = 0; it < m; ++it) {
                ma.key[it] = keys[i0 + it];
                ma.a_out[it] = SW + it * 2 * LN;
                ma.b_out[it] = SW + it * 2 * LN + LN;
                ma.init_b[it] = b[i0 + it];
            }
            ks_mac(c, ma, level, st);
            u64* p[2 * KS_MAX_ITEMS];
            const u64* base[2 * KS_MAX_ITEMS];
            u64* out[2 * KS_MAX_ITEMS];
            for (int it = 0; it < m; ++it) {
                p[2 * it] = AP + it * 2 * KN;
                p[2 * it + 1] = AP + it * 2 * KN + KN;
                base[2 * it] = out[2 * it] = SW + it * 2 * LN;
                base[2 * it + 1] = out[2 * it + 1] = SW + it * 2 * LN + LN;
            }
            ks_moddown_n(c, level, 2 * m, p, base, out, Tm, st);
        }
        // the automorphisms (the rotation's NTT-domain map)
        AutoItemsArgs aa{};
        aa.src = SW;
        for (int it = 0; it < m; ++it) {
            aa.galois[it] = galois[i0 + it] % (2 * N);
            aa.dst_a[it] = a_out[i0 + it];
            aa.dst_b[it] = b_out[i0 + it];
        }
        aa.L = L;
        aa.logN = c.logN;
        hipLaunchKernelGGL(k_automorphism_items, dim3((unsigned)(m * 2 * L * (N / KS_THREADS))), dim3(KS_THREADS),
                           0, st, aa);
        MI_HIP(hipGetLastError());
    });
}

void rotate_hoisted_batch(Context& c, int level, const u64* digits, const u64* b, int n, const u64* galois,
                          const u64* const* keys, u64* const* b_out, u64* const* a_out, bool montgomery,
                          hipStream_t s) {
    std::vector<const u64*> bs((size_t)std::max(n, 0), b);
    rotate_hoisted_items(c, level, digits, 0, n, bs.data(), n, galois, keys, b_out, a_out, montgomery, s);
}

// In-place rotations of independent ciphertexts at one level
// (ckks_rotate_inplace, ckks_rotation.cpp:41-96, for each): per chunk of up to
// KS_MAX_ITEMS, the key switches of all a run as one batch into a staging
// area (b enters as the switch's init_b: staged b = b + switched b, a
// assigned), and one launch applies each rotation's automorphism from the
// staging area back into the ciphertexts.
void rotate_batch(Context& c, int level, int n, u64* const* b, u64* const* a, const u64* galois,
                  const u64* const* keys, bool montgomery, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    if (n < 1) throw Error(-1, "need at least one rotation");
    const int L = level + 1;
    const u64 N = c.N;
    const long long LN = (long long)L * (long long)N;
    const int chunk = std::min(n, c.tune.ks_group);
    const size_t kw = ks_item_words(c, level);
    over_streams(c, s, (n + chunk - 1) / chunk, sizeof(u64) * (size_t)chunk * (kw + 2 * LN),
                 [&](hipStream_t st, u64* ws, int ci) {
        const int i0 = ci * chunk;
        const int m = std::min(chunk, n - i0);
        u64* SW = ws + (size_t)chunk * kw;  // per item: a' then b'
        KsItem items[KS_MAX_ITEMS];
        for (int it = 0; it < m; ++it) {
            u64* a_sw = SW + it * 2 * LN;
            u64* b_sw = a_sw + LN;
            items[it] = KsItem{a[i0 + it], keys[i0 + it], b_sw, a_sw, level, 1, 1, b[i0 + it]};
        }
        keyswitch_items_with(c, items, m, montgomery, ws, st);
        AutoItemsArgs aa{};
        aa.src = SW;
        for (int it = 0; it < m; ++it) {
            aa.galois[it] = galois[i0 + it] % (2 * N);
            aa.dst_a[it] = a[i0 + it];
            aa.dst_b[it] = b[i0 + it];
        }
        aa.L = L;
        aa.logN = c.logN;
        hipLaunchKernelGGL(k_automorphism_items, dim3((unsigned)(m * 2 * L * (N / KS_THREADS))), dim3(KS_THREADS),
                           0, st, aa);
        MI_HIP(hipGetLastError());
    });
}

// dst[k] = automorphism g of src[k] (L limbs each), for up to 2 KS_MAX_ITEMS polys
struct AutoListArgs {
    const u64* src[2 * KS_MAX_ITEMS];
    u64* dst[2 * KS_MAX_ITEMS];
    u64 galois;
    int L, logN;
};

__global__ void __launch_bounds__(KS_THREADS) k_automorphism_list(AutoListArgs a) {
    const u64 N = (u64)1 << a.logN;
    const int tps = (int)(N / KS_THREADS);
    const int tile = blockIdx.x % tps, rest = blockIdx.x / tps;
    const int l = rest % a.L, k = rest / a.L;
    const u32 i = (u32)tile * KS_THREADS + threadIdx.x;
    const long long off = (long long)l * N;
    a.dst[k][off + i] = a.src[k][off + galois_index(i, a.galois, a.logN)];
}

// One conjugation: both automorphisms in one launch into the workspace, from
// which the key switch reads its term and the b it adds.
void conjugate(Context& c, int level, u64* b, u64* a, const u64* key, bool montgomery, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    const int L = level + 1;
    const long long LN = (long long)L * (long long)c.N;
    u64* tmp = (u64*)c.workspace(s, sizeof(u64) * (2 * (size_t)LN + ks_item_words(c, level)));
    AutoListArgs al{};
    al.src[0] = a;
    al.src[1] = b;
    al.dst[0] = tmp;
    al.dst[1] = tmp + LN;
    al.galois = 2 * c.N - 1;
    al.L = L;
    al.logN = c.logN;
    hipLaunchKernelGGL(k_automorphism_list, dim3((unsigned)(2 * L * (c.N / KS_THREADS))), dim3(KS_THREADS), 0, s, al);
    MI_HIP(hipGetLastError());
    const KsItem it{tmp, key, b, a, level, 1, 1, tmp + LN};
    keyswitch_items_with(c, &it, 1, montgomery, tmp + 2 * LN, s);
}

void conjugate_batch(Context& c, int level, int n, u64* const* b, u64* const* a, const u64* key, bool montgomery,
                     hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    if (n < 1) return;
    const int L = level + 1;
    const u64 N = c.N;
    const long long LN = (long long)L * (long long)N;
    const u64 g = 2 * N - 1;
    // conjugated (a, b) of every ciphertext, live across the key-switch batch
    // (which uses the stream workspace itself)
    u64* tmp = (u64*)c.pool_alloc(sizeof(u64) * (size_t)n * 2 * LN);
    try {
        for (int i0 = 0; i0 < n; i0 += KS_MAX_ITEMS) {
            const int m = std::min(KS_MAX_ITEMS, n - i0);
            AutoListArgs al{};
            for (int it = 0; it < m; ++it) {
                al.src[2 * it] = a[i0 + it];
                al.src[2 * it + 1] = b[i0 + it];
                al.dst[2 * it] = tmp + (long long)(i0 + it) * 2 * LN;
                al.dst[2 * it + 1] = tmp + (long long)(i0 + it) * 2 * LN + LN;
            }
            al.galois = g;
            al.L = L;
            al.logN = c.logN;
            hipLaunchKernelGGL(k_automorphism_list, dim3((unsigned)(2 * m * L * (N / KS_THREADS))), dim3(KS_THREADS),
                               0, s, al);
            MI_HIP(hipGetLastError());
        }
        // (b, a) <- (sigma(b) + KS_b(sigma(a)), KS_a(sigma(a)))
        std::vector<KsItem> items;
        items.reserve(n);
        for (int k = 0; k < n; ++k) {
            const u64* ca = tmp + (long long)k * 2 * LN;
            items.push_back(KsItem{ca, key, b[k], a[k], level, 1, 1, ca + LN});
        }
        keyswitch_batch(c, items.data(), n, montgomery, s);
    } catch (...) {
        c.pool_release(tmp);
        throw;
    }
    c.pool_release(tmp);
}

void keyswitch_hoisted_qp(Context& c, int level, const u64* digits, const u64* key, const u64* b_q,
                          u64* b_qp, u64* a_qp, u64 galois, bool montgomery, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    MacArgs a = mac_args(c, level, digits, key, montgomery);
    a.qp_out = 1;
    a.b_out[0] = b_qp;
    a.a_out[0] = a_qp;
    a.galois = galois % (2 * c.N);
    a.init_b[0] = b_q;
    ks_mac(c, a, level, s);
}

void keyswitch_qp(Context& c, int level, const u64* key_term, const u64* key, u64* b_qp, u64* a_qp,
                  bool montgomery, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    const int L = level + 1, K = c.np, parts = c.parts(level);
    const u64 N = c.N;
    u64* C = (u64*)c.workspace(s, sizeof(u64) * (size_t)(L + parts * (L + K)) * N);
    u64* D = C + (size_t)L * N;
    ks_modup(c, level, key_term, D, C, s);
    MacArgs a = mac_args(c, level, D, key, montgomery);
    a.qp_out = 1;
    a.b_out[0] = b_qp;
    a.a_out[0] = a_qp;
    ks_mac(c, a, level, s);
}

void moddown_qp(Context& c, int level, u64* qp, hipStream_t s) {
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    const int L = level + 1;
    u64* T = (u64*)c.workspace(s, sizeof(u64) * (size_t)L * c.N);
    ks_moddown(c, level, qp + (size_t)L * c.N, nullptr, qp, nullptr, qp, nullptr, T, s);
}

}  // namespace mi
