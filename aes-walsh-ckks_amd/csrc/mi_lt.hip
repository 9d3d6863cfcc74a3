// BSGS linear-transform stage on the QP evaluator
// (ckks_apply_linear_transform_owned_stage_qp, ckks_linear_transform.cpp:1174-1407).
//
// With baby_steps = bs and the terms' diagonals d = g*bs + r:
//   baby[0]  = ([a;0], [b;0])                         (make_direct_input_qp, :487-532)
//   baby[r]  = hoisted QP rotation of (b, a) by r      (ckks_keyswitch.cpp:675-852)
//   inner_g  = sum_{terms of g} baby[r] * diag_t       (QP basis, per limb)
//   g = 0:     out += inner_0
//   g > 0:     KS = QP key switch of ModDown(inner_g.a) with the key of g*bs,
//              out.a += rot_{g*bs}(KS.a), out.b += rot_{g*bs}(KS.b + inner_g.b)
//              (automorphism_qp_pair_accumulate, :373-416)
//   result   = folded ModDown of out                  (moddown_qp_pair_to_q_eval, :641-718)
// The baby steps exist only inside the fused inner-product kernel, which reads
// the digits through each rotation's map (or, for many giant steps over
// integers alone, are written out for k_lt_inner_all).
#include "mi_ntt_kernels.hpp"

#include <algorithm>
#include <vector>

namespace mi {

constexpr int LT_THREADS = 256;
constexpr int LT_NB = 16;  // baby-step slots held in registers per launch (slot 0 = the input)
constexpr int LT_NG = 16;  // giant steps per launch

// Inner products of every giant step.  One block computes one giant step's
// sum for 256 coefficients of one limb of one ciphertext, streaming its (up
// to 16) baby/diagonal pairs: few registers, and a block touches only the
// memory of its own terms.  Block order (map_tile_g) puts the blocks of every
// giant step and ciphertext for one coefficient tile consecutively on one
// XCD, so the tile's baby steps (read once per giant step) and diagonals (read
// once per ciphertext) are served from that XCD's L2: HBM sees each baby step
// once per ciphertext and each diagonal once per batch.
struct LtAllArgs {
    const u64* diag[LT_NG * LT_NB];     // [giant][baby slot], null: no term
    const u64* in_a[KS_MAX_ITEMS];      // baby slot 0 (Q limbs; its P limbs are zero)
    const u64* in_b[KS_MAX_ITEMS];
    const u64* babies;                  // item i's baby s (s >= 1): a at babies +
    long long baby_item_stride;         //   i*item_stride + (s-1)*slot_stride, b T*N later
    long long baby_slot_stride;
    u64* out[LT_NG];                    // giant g of item i: a at out[g] + i*out_stride[g], b T*N later
    long long out_stride[LT_NG];
    int slot0;                          // baby slot of this launch's first term (multiple of 16)
    int nb, ng, accumulate;
    int items, L, K, nq, logN, pt_mont;
    const BasisConst* bc;
};

__global__ void __launch_bounds__(LT_THREADS) k_lt_inner_all(LtAllArgs a) {
    const u64 N = (u64)1 << a.logN;
    const int T = a.L + a.K;
    const int tps = (int)(N / LT_THREADS);
    // block -> (giant, item, slot, tile): giant fastest, then item, per XCD
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int g = local % a.ng, rest = local / a.ng;
    const int it = rest % a.items, tl = rest / a.items;
    const int tile = tl * 8 + xcd;
    const int slot = tile / tps;
    if (slot >= T) return;
    const long long i = (long long)(tile - slot * tps) * LT_THREADS + threadIdx.x;
    const int basis = slot < a.L ? slot : a.nq + (slot - a.L);
    const BasisConst b = a.bc[basis];
    const long long o = (long long)slot * N + i;
    const long long TN = (long long)T * N;
    // exact 128-bit sums: at most LT_NB = 16 products of residues below
    // 2^62 (plaintexts brought below q first) stay below 2^128; one reduction
    // at the end (REDC for Montgomery-form plaintexts, Barrett otherwise)
    // gives the canonical residue of the sum
    U128 sa{0, 0}, sb{0, 0};
    for (int r = 0; r < a.nb; ++r) {
        const u64* dp = a.diag[g * LT_NB + r];
        if (!dp) continue;
        const int sl = a.slot0 + r;
        u64 xa, xb;
        if (sl == 0) {
            if (slot >= a.L) continue;  // the input's P limbs are zero
            xa = a.in_a[it][o];
            xb = a.in_b[it][o];
        } else {
            const u64* p = a.babies + it * a.baby_item_stride + (long long)(sl - 1) * a.baby_slot_stride + o;
            xa = p[0];
            xb = p[TN];
        }
        const u64 d = reduce_4q(dp[o], b.q);
        mac128(sa, xa, d);
        mac128(sb, xb, d);
    }
    u64 ra, rb;
    if (a.pt_mont) {
        ra = redc128_any(sa.lo, sa.hi, b.q, b.qninv, b.mu_hi);
        rb = redc128_any(sb.lo, sb.hi, b.q, b.qninv, b.mu_hi);
    } else {
        ra = reduce128(sa.lo, sa.hi, b.q, b.mu_lo, b.mu_hi);
        rb = reduce128(sb.lo, sb.hi, b.q, b.mu_lo, b.mu_hi);
    }
    u64* pa = a.out[g] + it * a.out_stride[g] + o;
    u64* pb = pa + TN;
    *pa = a.accumulate ? add_mod(*pa, ra, b.q) : ra;
    *pb = a.accumulate ? add_mod(*pb, rb, b.q) : rb;
}

// Baby steps and inner products of the QP evaluator in one pass.  A thread
// forms, for one coefficient of one limb, the baby step of each rotation (the
// key product of the hoisted digits, read through the rotation's map, with the
// b term) and adds its product with every giant step's diagonal, so no baby
// step is written or read: at N = 2^16, 35 limbs, 15 rotations, 32 ciphertexts
// the separate passes moved 70 GB of babies and re-read digits.  IT ciphertexts
// share the loaded keys and diagonals and NG giant steps share the baby step;
// IT * NG = 16 keeps the sums in 64 registers.  The blocks of one tile for all
// ciphertexts follow each other on one XCD (map_tile): keys and diagonals come
// from memory once per launch, the digits of a limb's ciphertexts (2 MB each)
// stay in the Infinity Cache while its tiles run.
struct LtFusedArgs {
    const u64* diag[LT_NG * LT_NB];  // [giant][baby slot]; no term: a row of N zeros
    unsigned term[LT_NB];            // bit g: baby slot slot0 + r has a term of giant g
    const u64* key[LT_NB];           // baby slot slot0 + r
    u64 galois[LT_NB];
    const u64* in_a[KS_MAX_ITEMS];
    const u64* in_b[KS_MAX_ITEMS];
    const u64* digits;               // item i's [parts][T][N] at digits + i*digit_stride
    long long digit_stride;
    u64* out[LT_NG];                 // giant g of item i: a at out[g] + i*out_stride[g], b T*N later
    long long out_stride[LT_NG];
    int slot0, nb, ng, accumulate;
    int items, L, K, nq, logN, parts, mont, pt_mont;
    const BasisConst* bc;
};

// All words of a rotation are loaded before any is used, the diagonals without
// a branch (a missing term reads zeros): one wait per rotation instead of one
// per digit and giant step.
template <int NG, int IT, int PARTS>
__device__ __forceinline__ void lt_fused_fp(const LtFusedArgs& a, const BasisConst& b, int it0, int slot, long long i) {
    const u64 N = (u64)1 << a.logN;
    const int T = a.L + a.K, basis = slot < a.L ? slot : a.nq + (slot - a.L);
    const long long o = (long long)slot * N, to_a = (long long)(a.nq + a.K) * N;
    const FpMod m{b.qd, b.inv_d};
    double sa[IT][NG], sb[IT][NG];
#pragma unroll
    for (int t = 0; t < IT; ++t)
#pragma unroll
        for (int g = 0; g < NG; ++g) sa[t][g] = sb[t][g] = 0.0;
    int item[IT];
#pragma unroll
    for (int t = 0; t < IT; ++t) item[t] = it0 + t < a.items ? it0 + t : a.items - 1;  // past the end: a repeat, not stored
    for (int r = 0; r < a.nb; ++r) {
        u64 dw[NG];
        const unsigned term = a.term[r];
#pragma unroll
        for (int g = 0; g < NG; ++g) dw[g] = a.diag[g * LT_NB + r][((term >> g) & 1) ? o + i : i];
        double xa[IT], xb[IT];
        if (a.slot0 + r == 0) {
            if (slot >= a.L) continue;  // the input's P limbs are zero
#pragma unroll
            for (int t = 0; t < IT; ++t) {
                xa[t] = fp_from_u64(a.in_a[item[t]][o + i]);
                xb[t] = fp_from_u64(a.in_b[item[t]][o + i]);
            }
        } else {
            const u32 src = galois_index((u32)i, a.galois[r], a.logN);
            const u64* k = a.key[r] + (long long)basis * N + src;
            const u64* d = a.digits + o + src;
            u64 bw[IT];
#pragma unroll
            for (int t = 0; t < IT; ++t) {
                bw[t] = slot < a.L ? a.in_b[item[t]][o + src] : 0;
                xa[t] = xb[t] = 0.0;
            }
            // digits canonical, keys below 4q: each product at most 2q; three of
            // them (6q) between two reductions
            if constexpr (PARTS > 0) {
                u64 kw[PARTS][2], xw[PARTS][IT];
#pragma unroll
                for (int e = 0; e < PARTS; ++e) {
                    kw[e][0] = k[2LL * e * to_a];
                    kw[e][1] = k[(2LL * e + 1) * to_a];
#pragma unroll
                    for (int t = 0; t < IT; ++t) xw[e][t] = d[item[t] * a.digit_stride + (long long)e * T * N];
                }
#pragma unroll
                for (int e = 0; e < PARTS; ++e)
#pragma unroll
                    for (int t = 0; t < IT; ++t) {
                        const double x = fp_from_u64(xw[e][t]);
                        xb[t] += m.mulq(x, fp_from_u64(kw[e][0]));
                        xa[t] += m.mulq(x, fp_from_u64(kw[e][1]));
                        if (e == 2 && PARTS > 3) {
                            xb[t] = m.centred(xb[t]);
                            xa[t] = m.centred(xa[t]);
                        }
                    }
            } else {
                for (int e = 0; e < a.parts; ++e) {
                    const double kb = fp_from_u64(k[2LL * e * to_a]), ka = fp_from_u64(k[(2LL * e + 1) * to_a]);
#pragma unroll
                    for (int t = 0; t < IT; ++t) {
                        const double x = fp_from_u64(d[item[t] * a.digit_stride + (long long)e * T * N]);
                        xb[t] += m.centred(m.mulq(x, kb));
                        xa[t] += m.centred(m.mulq(x, ka));
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < IT; ++t) {
                if (a.mont) {
                    xb[t] = m.mul(xb[t], b.rinv_fp, b.rinv_fpq);
                    xa[t] = m.mul(xa[t], b.rinv_fp, b.rinv_fpq);
                } else if (PARTS == 0) {
                    xb[t] = m.centred(xb[t]);  // 16 digits reach 8q: no room for b
                }
                xb[t] = m.centred(xb[t] + fp_from_u64(bw[t]));
                xa[t] = m.centred(xa[t]);
            }
        }
        // |x| < q (the input) or q/2 (the others), diagonals below 4q: products
        // at most 2q or 5/4 q; four of them between two reductions, below 6q
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const double d = fp_from_u64(dw[g]);
#pragma unroll
            for (int t = 0; t < IT; ++t) {
                sa[t][g] += m.mulq(xa[t], d);
                sb[t][g] += m.mulq(xb[t], d);
            }
        }
        if ((r & 3) == 3) {
#pragma unroll
            for (int t = 0; t < IT; ++t)
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    sa[t][g] = m.centred(sa[t][g]);
                    sb[t][g] = m.centred(sb[t][g]);
                }
        }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        if (g >= a.ng) continue;
#pragma unroll
        for (int t = 0; t < IT; ++t) {
            if (it0 + t >= a.items) continue;
            double ra = sa[t][g], rb = sb[t][g];
            if (a.pt_mont) {
                ra = m.mul(ra, b.rinv_fp, b.rinv_fpq);
                rb = m.mul(rb, b.rinv_fp, b.rinv_fpq);
            }
            u64* pa = a.out[g] + (it0 + t) * a.out_stride[g] + o + i;
            u64* pb = pa + (long long)T * N;
            const u64 va = m.canonical(ra), vb = m.canonical(rb);
            *pa = a.accumulate ? add_mod(*pa, va, b.q) : va;
            *pb = a.accumulate ? add_mod(*pb, vb, b.q) : vb;
        }
    }
}

// Any modulus: canonical baby steps, exact 128-bit sums (at most 16 products
// of residues below 2^62), one ciphertext and the NG giant steps from g0 on at
// a time (a sum takes four registers).
template <int NG>
__device__ __forceinline__ void lt_fused_int(const LtFusedArgs& a, const BasisConst& b, int it, int g0, int slot,
                                             long long i) {
    const u64 N = (u64)1 << a.logN;
    const int T = a.L + a.K, basis = slot < a.L ? slot : a.nq + (slot - a.L);
    const long long o = (long long)slot * N, to_a = (long long)(a.nq + a.K) * N;
    U128 sa[NG], sb[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) sa[g] = sb[g] = U128{0, 0};
    const bool lazy = a.parts <= 3 && b.q < (1ull << 61);  // as in k_mac
    for (int r = 0; r < a.nb; ++r) {
        u64 xa, xb;
        if (a.slot0 + r == 0) {
            if (slot >= a.L) continue;
            xa = a.in_a[it][o + i];
            xb = a.in_b[it][o + i];
        } else {
            const u32 src = galois_index((u32)i, a.galois[r], a.logN);
            const u64* k = a.key[r] + (long long)basis * N + src;
            const u64* d = a.digits + it * a.digit_stride + o + src;
            U128 pa{0, 0}, pb{0, 0};
            for (int e = 0; e < a.parts; ++e) {
                u64 x = d[(long long)e * T * N], kb = k[2LL * e * to_a], ka = k[(2LL * e + 1) * to_a];
                if (!lazy) {
                    x = reduce_4q(x, b.q);
                    kb = reduce_4q(kb, b.q);
                    ka = reduce_4q(ka, b.q);
                }
                mac128(pb, x, kb);
                mac128(pa, x, ka);
            }
            pb.hi = reduce64(pb.hi, b.q, b.mu_hi);
            pa.hi = reduce64(pa.hi, b.q, b.mu_hi);
            xb = a.mont ? redc128(pb.lo, pb.hi, b.q, b.qninv) : barrett128(pb.lo, pb.hi, b.q, b.mu_lo, b.mu_hi);
            xa = a.mont ? redc128(pa.lo, pa.hi, b.q, b.qninv) : barrett128(pa.lo, pa.hi, b.q, b.mu_lo, b.mu_hi);
            if (slot < a.L) xb = add_mod(xb, a.in_b[it][o + src], b.q);
        }
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (!((a.term[r] >> (g0 + g)) & 1)) continue;
            const u64 d = reduce_4q(a.diag[(g0 + g) * LT_NB + r][o + i], b.q);
            mac128(sa[g], xa, d);
            mac128(sb[g], xb, d);
        }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        if (g0 + g >= a.ng) continue;
        u64 va, vb;
        if (a.pt_mont) {
            va = redc128_any(sa[g].lo, sa[g].hi, b.q, b.qninv, b.mu_hi);
            vb = redc128_any(sb[g].lo, sb[g].hi, b.q, b.qninv, b.mu_hi);
        } else {
            va = reduce128(sa[g].lo, sa[g].hi, b.q, b.mu_lo, b.mu_hi);
            vb = reduce128(sb[g].lo, sb[g].hi, b.q, b.mu_lo, b.mu_hi);
        }
        u64* pa = a.out[g0 + g] + it * a.out_stride[g0 + g] + o + i;
        u64* pb = pa + (long long)T * N;
        *pa = a.accumulate ? add_mod(*pa, va, b.q) : va;
        *pb = a.accumulate ? add_mod(*pb, vb, b.q) : vb;
    }
}

// PARTS = the digits (1 to 5), or 0: any number, one after the other.
template <int NG, int IT, int PARTS>
__global__ void __launch_bounds__(LT_THREADS) k_lt_fused(LtFusedArgs a) {
    const int tps = (1 << a.logN) / LT_THREADS;
    const TileMap tm = map_tile(blockIdx.x, (a.items + IT - 1) / IT, tps, a.L + a.K);
    if (!tm.valid) return;
    const long long i = (long long)tm.tile * LT_THREADS + threadIdx.x;
    const BasisConst b = a.bc[tm.slot < a.L ? tm.slot : a.nq + (tm.slot - a.L)];
    const int it0 = tm.item * IT;
    if (b.fp) {
        lt_fused_fp<NG, IT, PARTS>(a, b, it0, tm.slot, i);
    } else {
#pragma unroll 1
        for (int t = 0; t < IT && it0 + t < a.items; ++t)
#pragma unroll 1
            for (int g0 = 0; g0 < a.ng; g0 += 8) lt_fused_int<(NG < 8 ? NG : 8)>(a, b, it0 + t, g0, tm.slot, i);
    }
}

// Contexts whose moduli are all integers: one ciphertext per workgroup, at most
// NG giant steps.  Nothing is shared between ciphertexts here, and the forms
// above run two or four of them one after the other.  8 baby steps, us, separate
// baby steps / the forms above / this one: N = 2^15, 12 limbs of 60 bits, 6
// digits, one giant step, 5 ciphertexts 641 / 937 / 529; 3 digits, 4 giant
// steps, 16 ciphertexts 3464 / 3396 / 2904; N = 2^16, 30 limbs, 2 giant steps, 5
// ciphertexts 3564 / 4572 / 3021.
template <int NG>
__global__ void __launch_bounds__(LT_THREADS) k_lt_int(LtFusedArgs a) {
    const int tps = (1 << a.logN) / LT_THREADS;
    const TileMap tm = map_tile(blockIdx.x, a.items, tps, a.L + a.K);
    if (!tm.valid) return;
    const long long i = (long long)tm.tile * LT_THREADS + threadIdx.x;
    const BasisConst b = a.bc[tm.slot < a.L ? tm.slot : a.nq + (tm.slot - a.L)];
    lt_fused_int<NG>(a, b, tm.item, 0, tm.slot, i);
}

static u64 powmod_u64(u64 a, u64 e, u64 m) {
    unsigned __int128 r = 1, x = a % m;
    while (e) {
        if (e & 1) r = r * x % m;
        x = x * x % m;
        e >>= 1;
    }
    return (u64)r;
}

// Galois element of a slot rotation (rotation_key_generation.cpp:73-78):
// 5^(r mod N/2) mod 2N.
u64 rotation_galois(u64 N, long long rotation) {
    const long long slots = (long long)(N >> 1);
    long long r = rotation % slots;
    if (r < 0) r += slots;
    return powmod_u64(5, (u64)r, N << 1);
}

namespace {

// compile_linear_transform_stage_metadata (ckks_linear_transform.cpp:720-756)
// plus the key lookups: baby steps in use get slots 1.. in order of first use
// (slot 0 is the input itself); giant steps in use are listed in order.
struct Compiled {
    int bs = 0, nslots = 1, ngp = 0;
    bool g0 = false;
    std::vector<int> baby_slot;            // rotation r < bs -> slot, -1 unused
    std::vector<int> glist;                // giant indices in use, ascending
    std::vector<const u64*> table;         // [giant index][slot] diagonal
    std::vector<const u64*> baby_key;      // [slot]
    std::vector<u64> baby_gal;             // [slot]
    std::vector<const u64*> giant_key;     // [giant index]
};

Compiled compile_stage(const Context& c, const LtStage& st, bool q_eval) {
    const int level = st.level;
    if (level < 0 || level >= c.nq) throw Error(-1, "invalid ciphertext level");
    if (st.nterms < 1 || st.baby_steps < 1 || st.slots < 1)
        throw Error(-1, "need nterms >= 1, baby_steps >= 1, slots >= 1");
    if (!st.diag_idx || !st.diags) throw Error(-1, "null pointer argument");
    if (st.nkeys > 0 && (!st.key_rot || !st.keys)) throw Error(-1, "null key table");
    Compiled k;
    const int bs = k.bs = st.baby_steps;
    const int giants = (st.slots + bs - 1) / bs;
    k.baby_slot.assign(bs, -1);
    k.baby_slot[0] = 0;
    std::vector<int> gidx(giants, -1);
    for (int t = 0; t < st.nterms; ++t) {
        const long long d = st.diag_idx[t];
        if (d < 0) throw Error(-1, "diagonal indices must be non-negative");
        if (!st.diags[t]) throw Error(-1, "null diagonal");
        if (d / bs >= giants) {
            // the Q evaluator's validation (:758-814) rejects such a term;
            // the QP evaluator leaves it out
            if (q_eval) throw Error(-1, "diagonal index exceeds slot count");
            continue;
        }
        const int r = (int)(d % bs), g = (int)(d / bs);
        if (k.baby_slot[r] < 0) k.baby_slot[r] = k.nslots++;
        if (gidx[g] < 0) {
            gidx[g] = 0;
            k.glist.push_back(g);
        }
    }
    if (k.glist.empty()) throw Error(-1, "no diagonal falls inside the slot range");
    std::sort(k.glist.begin(), k.glist.end());
    for (size_t j = 0; j < k.glist.size(); ++j) gidx[k.glist[j]] = (int)j;
    k.g0 = k.glist[0] == 0;
    k.ngp = (int)k.glist.size() - (k.g0 ? 1 : 0);
    k.table.assign(k.glist.size() * (size_t)k.nslots, nullptr);
    for (int t = 0; t < st.nterms; ++t) {
        const long long d = st.diag_idx[t];
        if (d / bs >= giants) continue;
        const u64*& e = k.table[(size_t)gidx[d / bs] * k.nslots + k.baby_slot[d % bs]];
        if (e) throw Error(-1, "duplicate diagonal index " + std::to_string(d));
        e = st.diags[t];
    }
    auto key_for = [&](long long r) -> const u64* {
        for (int i = 0; i < st.nkeys; ++i)
            if (st.key_rot[i] == r) {
                if (!st.keys[i]) throw Error(-1, "null rotation key");
                return st.keys[i];
            }
        throw Error(-1, "missing rotation key for step " + std::to_string(r));
    };
    // every key is looked up before any work is queued
    k.baby_key.assign(k.nslots, nullptr);
    k.baby_gal.assign(k.nslots, 0);
    for (int r = 1; r < bs; ++r)
        if (k.baby_slot[r] > 0) {
            k.baby_key[k.baby_slot[r]] = key_for(r);
            k.baby_gal[k.baby_slot[r]] = rotation_galois(c.N, r);
        }
    k.giant_key.assign(k.glist.size(), nullptr);
    for (size_t j = 0; j < k.glist.size(); ++j)
        if (k.glist[j] > 0) k.giant_key[j] = key_for((long long)k.glist[j] * bs);
    return k;
}

// Inner products of every giant step for m items.  Giant 0 goes to out0 +
// i*out0_stride, giant j > 0 (in use order) to outg + (j-1)*outg_giant +
// i*outg_item; K = 0 for the Q evaluator.
void launch_inner(Context& c, const Compiled& k, const LtStage& st, int m, int K, const u64* const* a,
                  const u64* const* b, const u64* babies, long long baby_item, long long baby_slot, u64* out0,
                  long long out0_stride, u64* outg, long long outg_giant, long long outg_item, hipStream_t s) {
    const int L = st.level + 1, T = L + K;
    const int tps = (int)(c.N / LT_THREADS);
    for (int s0 = 0; s0 < k.nslots; s0 += LT_NB) {
        for (size_t gk0 = 0; gk0 < k.glist.size(); gk0 += LT_NG) {
            LtAllArgs ia{};
            ia.nb = std::min(LT_NB, k.nslots - s0);
            ia.ng = (int)std::min<size_t>(LT_NG, k.glist.size() - gk0);
            ia.slot0 = s0;
            for (int g = 0; g < ia.ng; ++g) {
                const size_t gk = gk0 + g;
                for (int r = 0; r < ia.nb; ++r) ia.diag[g * LT_NB + r] = k.table[gk * k.nslots + s0 + r];
                if (k.glist[gk] == 0) {
                    ia.out[g] = out0;
                    ia.out_stride[g] = out0_stride;
                } else {
                    ia.out[g] = outg + (long long)(gk - (k.g0 ? 1 : 0)) * outg_giant;
                    ia.out_stride[g] = outg_item;
                }
            }
            for (int it = 0; it < m; ++it) {
                ia.in_a[it] = a[it];
                ia.in_b[it] = b[it];
            }
            ia.babies = babies;
            ia.baby_item_stride = baby_item;
            ia.baby_slot_stride = baby_slot;
            ia.accumulate = s0 > 0 ? 1 : 0;
            ia.items = m;
            ia.L = L;
            ia.K = K;
            ia.nq = c.nq;
            ia.logN = c.logN;
            ia.pt_mont = st.pt_montgomery ? 1 : 0;
            ia.bc = c.d_bc;
            hipLaunchKernelGGL(k_lt_inner_all, dim3(tile_grid(m * ia.ng, tps, T)), dim3(LT_THREADS), 0, s, ia);
            MI_HIP(hipGetLastError());
        }
    }
}

// Baby steps and inner products of m items from their hoisted digits; outputs
// as launch_inner.
void launch_fused(Context& c, const Compiled& k, const LtStage& st, int m, const u64* const* a, const u64* const* b,
                  const u64* digits, long long dstride, u64* out0, long long out0_stride, u64* outg,
                  long long outg_giant, long long outg_item, hipStream_t s) {
    const int L = st.level + 1, T = L + c.np;
    const int tps = (int)(c.N / LT_THREADS);
    const bool integer = c.integer_only();
    const size_t most = integer ? 8 : LT_NG;
    for (int s0 = 0; s0 < k.nslots; s0 += LT_NB) {
        for (size_t gk0 = 0; gk0 < k.glist.size(); gk0 += most) {
            LtFusedArgs f{};
            f.nb = std::min(LT_NB, k.nslots - s0);
            f.ng = (int)std::min<size_t>(most, k.glist.size() - gk0);
            f.slot0 = s0;
            for (int r = 0; r < f.nb; ++r) {
                f.key[r] = k.baby_key[s0 + r];
                f.galois[r] = k.baby_gal[s0 + r];
            }
            for (const u64*& d : f.diag) d = c.d_zero;
            for (int g = 0; g < f.ng; ++g) {
                const size_t gk = gk0 + g;
                for (int r = 0; r < f.nb; ++r) {
                    const u64* d = k.table[gk * k.nslots + s0 + r];
                    f.diag[g * LT_NB + r] = d ? d : c.d_zero;
                    if (d) f.term[r] |= 1u << g;
                }
                const bool first = k.glist[gk] == 0;
                f.out[g] = first ? out0 : outg + (long long)(gk - (k.g0 ? 1 : 0)) * outg_giant;
                f.out_stride[g] = first ? out0_stride : outg_item;
            }
            for (int it = 0; it < m; ++it) {
                f.in_a[it] = a[it];
                f.in_b[it] = b[it];
            }
            f.digits = digits;
            f.digit_stride = dstride;
            f.accumulate = s0 > 0 ? 1 : 0;
            f.items = m;
            f.L = L;
            f.K = c.np;
            f.nq = c.nq;
            f.logN = c.logN;
            f.parts = c.parts(st.level);
            f.mont = st.montgomery ? 1 : 0;
            f.pt_mont = st.pt_montgomery ? 1 : 0;
            f.bc = c.d_bc;
            if (integer) {
                const dim3 grid(tile_grid(m, tps, T));
                if (f.ng <= 4) hipLaunchKernelGGL(k_lt_int<4>, grid, dim3(LT_THREADS), 0, s, f);
                else hipLaunchKernelGGL(k_lt_int<8>, grid, dim3(LT_THREADS), 0, s, f);
                MI_HIP(hipGetLastError());
                continue;
            }
            // several ciphertexts: the fewest giant steps that hold f.ng, and with
            // them as many ciphertexts; one: 16 giant steps whatever f.ng is
#define MI_LT_FUSED(NG, IT, PARTS)                                                                     \
    hipLaunchKernelGGL((k_lt_fused<NG, IT, PARTS>), dim3(tile_grid((m + IT - 1) / IT, tps, T)),        \
                       dim3(LT_THREADS), 0, s, f)
#define MI_LT_FUSED_P(PARTS)                                                                           \
    if (f.ng <= 4 && m > 1) MI_LT_FUSED(4, 4, PARTS);                                                  \
    else if (f.ng <= 8 && m > 1) MI_LT_FUSED(8, 2, PARTS);                                             \
    else MI_LT_FUSED(16, 1, PARTS);
            switch (f.parts) {
                case 1: MI_LT_FUSED_P(1) break;
                case 2: MI_LT_FUSED_P(2) break;
                case 3: MI_LT_FUSED_P(3) break;
                case 4: MI_LT_FUSED_P(4) break;
                case 5: MI_LT_FUSED_P(5) break;
                default: MI_LT_FUSED_P(0)
            }
#undef MI_LT_FUSED_P
#undef MI_LT_FUSED
            MI_HIP(hipGetLastError());
        }
    }
}

void check_batch(int n, const u64* const* a, const u64* const* b, u64* const* a_out, u64* const* b_out) {
    if (n < 1 || !a || !b || !a_out || !b_out) throw Error(-1, "null pointer argument");
    for (int i = 0; i < n; ++i)
        if (!a[i] || !b[i] || !a_out[i] || !b_out[i]) throw Error(-1, "null pointer argument");
}

}  // namespace

void linear_transform_qp_batch(Context& c, const LtStage& st, int n, const u64* const* a,
                               const u64* const* b, u64* const* a_out, u64* const* b_out, hipStream_t s) {
    const Compiled k = compile_stage(c, st, false);
    check_batch(n, a, b, a_out, b_out);
    const int level = st.level;
    const int L = level + 1, K = c.np, T = L + K, parts = c.parts(level);
    const u64 N = c.N;
    const long long W = (long long)T * (long long)N, LN = (long long)L * (long long)N;
    const int nbaby = k.nslots - 1, ngp = k.ngp;

    // Integers alone and more than 8 giant steps: the baby steps are written once
    // and read by every giant step, unless the batch is small.  The fused kernel
    // holds 8 steps' sums (16 took up to 7 % longer) and forms each baby step again
    // for the next 8, which costs less than the extra launches up to some 850,000
    // coefficients.  16 baby and 16 giant steps of 60 bits, us, separate / fused:
    // N = 2^14, 10 limbs, 4 digits, 1, 5 and 16 ciphertexts (164 k, 819 k, 2.6 M)
    // 1866 / 1562, 2709 / 2667, 5235 / 5522; N = 2^15, 14 limbs, 6 digits, 1, 2 and
    // 5 (459 k, 918 k, 2.3 M) 2510 / 2473, 3247 / 3397, 5866 / 6375; N = 2^16, 40
    // limbs, 3 digits, 1 (2.6 M) 6223 / 6509.
    const bool separate = nbaby > 0 && k.glist.size() > 8 && n * W > 850000 && c.integer_only();

    // per-item scratch: digits | C | babies (a, b; separate) | out (a, b) | giant
    // inners (a, b) | ModDown temp
    const long long dw = (long long)parts * W, bw = separate ? 2 * (long long)nbaby * W : 0;
    const long long item_words = dw + LN + bw + 2 * W + 2 * (long long)ngp * W + 2 * LN;
    const long long budget_words = (32LL << 30) / 8;
    int chunk = (int)std::min<long long>(KS_MAX_ITEMS, std::max<long long>(1, budget_words / item_words));
    chunk = std::min(chunk, n);
    u64* ws = (u64*)c.workspace(s, sizeof(u64) * (size_t)(item_words * chunk));

    for (int i0 = 0; i0 < n; i0 += chunk) {
        const int m = std::min(chunk, n - i0);
        u64* D = ws;
        u64* C = D + m * dw;
        u64* BAB = C + m * LN;
        u64* OAB = BAB + m * bw;
        u64* IAB = OAB + m * 2 * W;
        u64* Tm = IAB + m * 2 * (long long)ngp * W;
        auto inner = [&](int it, int gp) { return IAB + it * 2LL * ngp * W + (long long)gp * 2 * W; };
        auto outp = [&](int it) { return OAB + it * 2 * W; };

        // one hoisted ModUp, then the baby steps (hoisted QP rotations, :675-852,
        // b added in the Q limbs) and every giant step's inner product
        if (nbaby > 0) ks_modup_n(c, level, m, a + i0, D, dw, C, s);
        if (separate) {
            // the baby steps' key products are independent (each writes its
            // own slot from the shared digits): spread over the streams
            over_streams(c, s, nbaby, 0, [&](hipStream_t bst, u64*, int i) {
                MacArgs ma = mac_args(c, level, D, k.baby_key[i + 1], st.montgomery != 0);
                ma.items = m;
                ma.digits_stride = dw;
                ma.qp_out = 1;
                ma.galois = k.baby_gal[i + 1];
                for (int it = 0; it < m; ++it) {
                    ma.key[it] = k.baby_key[i + 1];
                    ma.a_out[it] = BAB + it * bw + i * 2LL * W;
                    ma.b_out[it] = ma.a_out[it] + W;
                    ma.init_b[it] = b[i0 + it];
                }
                ks_mac(c, ma, level, bst);
            });
            launch_inner(c, k, st, m, K, a + i0, b + i0, BAB, bw, 2 * W, OAB, 2 * W, IAB, 2 * W, 2LL * ngp * W, s);
        } else {
            launch_fused(c, k, st, m, a + i0, b + i0, D, dw, OAB, 2 * W, IAB, 2 * W, 2LL * ngp * W, s);
        }

        // giant steps > 0: key term = ModDown(inner.a); QP switch; rotate-accumulate
        // with inner.b (automorphism_qp_pair_accumulate, :373-416)
        bool have_out = k.g0;
        u64* p[2 * KS_MAX_ITEMS];
        const u64* base[2 * KS_MAX_ITEMS];
        u64* outs[2 * KS_MAX_ITEMS];
        const u64* kt[KS_MAX_ITEMS];
        for (int gp = 0; gp < ngp; ++gp) {
            const size_t gk = (size_t)gp + (k.g0 ? 1 : 0);
            for (int it = 0; it < m; ++it) {
                p[it] = inner(it, gp) + LN;
                base[it] = outs[it] = inner(it, gp);
                kt[it] = inner(it, gp);
            }
            ks_moddown_n(c, level, m, p, base, outs, Tm, s);
            ks_modup_n(c, level, m, kt, D, dw, C, s);
            MacArgs ma = mac_args(c, level, D, k.giant_key[gk], st.montgomery != 0);
            ma.items = m;
            ma.digits_stride = dw;
            ma.qp_out = 1;
            ma.galois = rotation_galois(N, (long long)k.glist[gk] * k.bs);
            ma.accumulate = have_out ? 1 : 0;
            for (int it = 0; it < m; ++it) {
                ma.key[it] = k.giant_key[gk];
                ma.a_out[it] = outp(it);
                ma.b_out[it] = outp(it) + W;
                ma.add_b[it] = inner(it, gp) + W;
            }
            ks_mac(c, ma, level, s);
            have_out = true;
        }

        // result = folded ModDown of out (moddown_qp_pair_to_q_eval, :641-718)
        for (int it = 0; it < m; ++it) {
            p[2 * it] = outp(it) + LN;
            p[2 * it + 1] = outp(it) + W + LN;
            base[2 * it] = outp(it);
            base[2 * it + 1] = outp(it) + W;
            outs[2 * it] = a_out[i0 + it];
            outs[2 * it + 1] = b_out[i0 + it];
        }
        ks_moddown_n(c, level, 2 * m, p, base, outs, Tm, s);
    }
}

void linear_transform_q_batch(Context& c, const LtStage& st, int n, const u64* const* a,
                              const u64* const* b, u64* const* a_out, u64* const* b_out, hipStream_t s) {
    const Compiled k = compile_stage(c, st, true);
    check_batch(n, a, b, a_out, b_out);
    const int level = st.level;
    const int L = level + 1, K = c.np, parts = c.parts(level);
    const u64 N = c.N;
    const long long LN = (long long)L * (long long)N, KN = (long long)K * (long long)N;
    const int nbaby = k.nslots - 1, ngp = k.ngp;
    const long long dw = (long long)parts * (L + K) * (long long)N;

    // per-item scratch: digits | C | P accumulators | ModDown temp | switched
    // pair | babies [slot][item] | out | giant inners [giant][item]
    const long long item_words = dw + LN + 2 * KN + 2 * LN + 2 * LN + 2 * (long long)nbaby * LN + 2 * LN +
                                 2 * (long long)ngp * LN;
    const long long budget_words = (32LL << 30) / 8;
    int chunk = (int)std::min<long long>(KS_MAX_ITEMS, std::max<long long>(1, budget_words / item_words));
    chunk = std::min(chunk, n);
    // Folded, the baby steps of all ciphertexts are one batch and so are the
    // giant steps' switches, ck (step, ciphertext) pairs at a time: a few
    // ciphertexts' single steps leave most of the chip idle.  Each pair takes
    // step_words of scratch, so ck ends where a pass over its two polynomials
    // has 2^25 words (8192 workgroups, 32 per CU) and where the budget does:
    // 16 pairs of 13 limbs at N = 2^15 (3328 workgroups) took 5 % longer than
    // 32, 8 pairs of 30 limbs at N = 2^16 (7680) 1 %, and 32 of those would
    // hold 4.9 GB.
    const long long step_words = dw + LN + 2 * KN + 2 * LN + 2 * LN;  // digits | C | P accumulators | temp | switched
    const bool fold = parts <= 3 && c.fuse_mac;
    int ck = chunk;
    if (fold) {
        const long long pairs = (long long)chunk * std::max(1, std::max(nbaby, ngp));
        const long long fill = ((1LL << 25) + 2 * LN - 1) / (2 * LN);
        const long long fit = chunk + std::max(0LL, budget_words - item_words * chunk) / step_words;
        ck = std::max(chunk, (int)std::min({(long long)KS_MAX_ITEMS, pairs, fill, fit}));
    }
    auto bytes = [&](int k) { return sizeof(u64) * (size_t)(step_words * k + (item_words - step_words) * chunk); };
    bool whole = true;
    u64* ws = (u64*)c.workspace_up_to(s, bytes(ck), bytes(chunk), &whole);
    if (!whole) ck = chunk;

    for (int i0 = 0; i0 < n; i0 += chunk) {
        const int m = std::min(chunk, n - i0);
        u64* D = ws;
        u64* C = D + ck * dw;
        u64* AP = C + ck * LN;
        u64* Tm = AP + ck * 2 * KN;
        u64* SW = Tm + ck * 2 * LN;
        u64* BQ = SW + ck * 2 * LN;
        u64* OQ = BQ + m * 2 * (long long)nbaby * LN;
        u64* IQ = OQ + m * 2 * LN;
        u64* p[2 * KS_MAX_ITEMS];
        const u64* base[2 * KS_MAX_ITEMS];
        u64* outs[2 * KS_MAX_ITEMS];

        // key switch of m key terms into SW (a at +0, b at +LN per item, b
        // starting from b_init), modes Assign: the hoisted or full switch
        // of ckks_hybrid_key_switch_(hoisted_)inplace
        auto mac_moddown = [&](const u64* key, const u64* const* b_init) {
            MacArgs ma = mac_args(c, level, D, key, st.montgomery != 0);
            ma.items = m;
            ma.digits_stride = dw;
            ma.accp = AP;
            ma.accp_stride = 2 * KN;
            ma.b_mode = 1;
            ma.a_mode = 1;
            for (int it = 0; it < m; ++it) {
                ma.key[it] = key;
                ma.a_out[it] = SW + it * 2 * LN;
                ma.b_out[it] = SW + it * 2 * LN + LN;
                ma.init_b[it] = b_init[it];
            }
            ks_mac(c, ma, level, s);
            for (int it = 0; it < m; ++it) {
                p[2 * it] = AP + it * 2 * KN;
                p[2 * it + 1] = AP + it * 2 * KN + KN;
                base[2 * it] = outs[2 * it] = SW + it * 2 * LN;
                base[2 * it + 1] = outs[2 * it + 1] = SW + it * 2 * LN + LN;
            }
            ks_moddown_n(c, level, 2 * m, p, base, outs, Tm, s);
        };

        // baby steps: hoisted rotations in Q (ckks_hybrid_key_switch_hoisted_inplace
        // with b Add and a Assign, then the automorphism), [slot][item] layout
        if (nbaby > 0) {
            ks_modup_n(c, level, m, a + i0, D, dw, C, s);
            // (slot, ciphertext) pairs in order, each stored through its rotation's map
            for (int j0 = 0; fold && j0 < nbaby * m; j0 += ck) {
                const int n1 = std::min(ck, nbaby * m - j0);
                KsItem items[KS_MAX_ITEMS];
                for (int e = 0; e < n1; ++e) {
                    const int sl = (j0 + e) / m + 1, it = (j0 + e) % m;
                    u64* o = BQ + ((long long)(sl - 1) * m + it) * 2 * LN;
                    items[e] = KsItem{nullptr, k.baby_key[sl], o + LN, o, level, 1, 1, b[i0 + it], k.baby_gal[sl]};
                }
                ks_moddown_mac(c, level, n1, items, D, dw, AP, Tm, st.montgomery != 0, s, j0, m);
            }
            for (int sl = 1; !fold && sl < k.nslots; ++sl) {
                mac_moddown(k.baby_key[sl], b + i0);
                automorphism(c, L, k.baby_gal[sl], SW, BQ + (long long)(sl - 1) * m * 2 * LN, 2 * m, LN, LN, s);
            }
        }

        launch_inner(c, k, st, m, 0, a + i0, b + i0, BQ, 2 * LN, (long long)m * 2 * LN, OQ, 2 * LN, IQ,
                     (long long)m * 2 * LN, 2 * LN, s);

        // giant steps > 0: rotate each inner sum by a full key switch
        // (ckks_rotate_inplace: switch a, then the automorphism) and add
        bool have_out = k.g0;
        for (int j0 = 0; fold && j0 < ngp * m; j0 += ck) {
            const int n1 = std::min(ck, ngp * m - j0);
            const u64* kt[KS_MAX_ITEMS];
            KsItem items[KS_MAX_ITEMS];
            for (int e = 0; e < n1; ++e) {
                const size_t gk = (size_t)((j0 + e) / m) + (k.g0 ? 1 : 0);
                const u64* in = IQ + (long long)(j0 + e) * 2 * LN;
                u64* o = SW + (long long)e * 2 * LN;
                kt[e] = in;
                items[e] = KsItem{nullptr, k.giant_key[gk], o + LN, o, level, 1, 1, in + LN,
                                  rotation_galois(N, (long long)k.glist[gk] * k.bs)};
            }
            ks_modup_n(c, level, n1, kt, D, dw, C, s);
            ks_moddown_mac(c, level, n1, items, D, dw, AP, Tm, st.montgomery != 0, s);
            // the switched sums of one giant step at a time onto the ciphertexts
            for (int e = 0; e < n1;) {
                const int it0 = (j0 + e) % m, run = std::min(n1 - e, m - it0);
                u64* dst[2 * KS_MAX_ITEMS];
                const u64* src[2 * KS_MAX_ITEMS];
                for (int r = 0; r < 2 * run; ++r) {
                    dst[r] = OQ + ((long long)it0 * 2 + r) * LN;
                    src[r] = SW + ((long long)e * 2 + r) * LN;
                }
                const bool first = !k.g0 && (j0 + e) / m == 0;
                pair_list_op(c, first ? 0 : 1, level, dst, src, 2 * run, nullptr, s);  // copy or add
                e += run;
            }
        }
        for (int gp = 0; !fold && gp < ngp; ++gp) {
            const size_t gk = (size_t)gp + (k.g0 ? 1 : 0);
            u64* in = IQ + (long long)gp * m * 2 * LN;
            const u64* kt[KS_MAX_ITEMS];
            const u64* bi[KS_MAX_ITEMS];
            for (int it = 0; it < m; ++it) {
                kt[it] = in + it * 2 * LN;
                bi[it] = in + it * 2 * LN + LN;
            }
            ks_modup_n(c, level, m, kt, D, dw, C, s);
            mac_moddown(k.giant_key[gk], bi);
            automorphism_acc(c, L, rotation_galois(N, (long long)k.glist[gk] * k.bs), SW, OQ, 2 * m, LN, LN,
                             have_out, s);
            have_out = true;
        }
        u64* dst[2 * KS_MAX_ITEMS];
        const u64* src[2 * KS_MAX_ITEMS];
        for (int it = 0; it < m; ++it) {
            dst[2 * it] = a_out[i0 + it];
            dst[2 * it + 1] = b_out[i0 + it];
            src[2 * it] = OQ + it * 2 * LN;
            src[2 * it + 1] = src[2 * it] + LN;
        }
        pair_list_op(c, 0, level, dst, src, 2 * m, nullptr, s);  // copy
    }
}

void linear_transform_qp(Context& c, const LtStage& st, const u64* a, const u64* b, u64* a_out,
                         u64* b_out, hipStream_t s) {
    linear_transform_qp_batch(c, st, 1, &a, &b, &a_out, &b_out, s);
}

}  // namespace mi
