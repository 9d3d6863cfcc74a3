// Steps of the folded ModDown shared by mi_moddown.hip and mi_moddown_mac.hip.
#pragma once
#include "mi_ntt_kernels.hpp"

namespace mi {

constexpr int KS_THREADS = 256;
constexpr int MAX_ALPHA = 16;  // digit width (or special moduli) held in registers

#define MI_NS_CASES(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16)

// second inverse pass over the P limbs (p[k]: K limbs of poly k)
void moddown_p_cols(const Context& c, int npoly, u64* const* p, hipStream_t s);
// contributions of the coefficient-domain P limbs to every Q limb: T [npoly][L][N]
void moddown_contrib(const Context& c, int level, int npoly, u64* const* p, u64* T, hipStream_t s);
// first forward pass over the contributions
void moddown_contrib_cols(const Context& c, int level, int npoly, u64* T, hipStream_t s);

}  // namespace mi
