// Batched negacyclic NTT kernels (two passes over HBM, see mi_ntt_core.hpp).
//
// Forward = reference ntt_forward_dit2 (ntt.cpp:235-297): column pass runs
// global stages 0..n1-1, row pass runs n1..n-1 and reduces to [0, q).
// Inverse = reference ntt_inverse_dif2 (ntt.cpp:331-386): row pass runs the
// distance 1..R2/2 stages, column pass the rest and multiplies by N^-1.
//
// The kernels are templated on a Job that maps the batch's limb k to a view
// with basis(), load(i) and store(i, v); plain in-place NTTs and the fused
// rescale / key-switch steps (prologue computes the input, epilogue combines
// the output) share the same butterfly code.
#include "mi_ntt_kernels.hpp"

namespace mi {

namespace {
template <bool FWD, bool ROWS, Arith A>
void one_limb(const Context& c, const PlainJob& job, int count, hipStream_t s) {
    if constexpr (ROWS) launch_rows<FWD, 1, false, A>(c, job, count, s);
    else launch_cols<FWD, 1, false, A>(c, job, count, s);
}

template <bool FWD, bool ROWS>
void plain_pass(const Context& c, int variant, const PlainJob& job, int count, hipStream_t s) {
    switch (variant) {
        case 2:
            if constexpr (ROWS) launch_rows<FWD, 2, false>(c, job, count, s);
            else launch_cols<FWD, 2, false>(c, job, count, s);
            break;
        case 3:
            if constexpr (ROWS) launch_rows<FWD, 1, true>(c, job, count, s);
            else launch_cols<FWD, 1, true>(c, job, count, s);
            break;
        default: {
            int fp = 0;
            for (int l = 0; l < job.b.lpp; ++l) fp += c.h_bc[job.b.basis0 + l].fp ? 1 : 0;
            if (fp == 0) one_limb<FWD, ROWS, Arith::Int>(c, job, count, s);
            else if (fp == job.b.lpp) one_limb<FWD, ROWS, Arith::Fp>(c, job, count, s);
            else one_limb<FWD, ROWS, Arith::Both>(c, job, count, s);
        }
    }
}
}  // namespace

void launch_plain_pass(const Context& c, bool fwd, bool rows, int variant, const PlainJob& job, int count,
                       hipStream_t s) {
    if (fwd && rows) plain_pass<true, true>(c, variant, job, count, s);
    else if (fwd) plain_pass<true, false>(c, variant, job, count, s);
    else if (rows) plain_pass<false, true>(c, variant, job, count, s);
    else plain_pass<false, false>(c, variant, job, count, s);
}

void ntt_forward(const Context& c, const LimbBatch& b, hipStream_t s) {
    if (b.count <= 0) return;
    const PlainJob j = plain_job(b, c.N);
    run_ntt_fwd(c, j, j, b.count, s);
}

void ntt_inverse(const Context& c, const LimbBatch& b, hipStream_t s) {
    if (b.count <= 0) return;
    const PlainJob j = plain_job(b, c.N);
    run_ntt_inv(c, j, j, b.count, s);
}

}  // namespace mi
