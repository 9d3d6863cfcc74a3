// Steps of the folded ModDown shared by mi_moddown.hip and mi_moddown_mac.hpp.
#pragma once
#include "mi_ntt_kernels.hpp"

namespace mi {

constexpr int KS_THREADS = 256;
constexpr int MAX_ALPHA = 16;  // digit width (or special moduli) held in registers

// second inverse pass over the P limbs (p[k]: K limbs of poly k)
void moddown_p_cols(const Context& c, int npoly, u64* const* p, hipStream_t s);
// contributions of the coefficient-domain P limbs to every Q limb and their
// first forward pass: T [npoly][L][N]
void moddown_ext_cols(const Context& c, int level, int npoly, u64* const* p, u64* T, hipStream_t s);

// ModDown with the key inner product of 1 to 3 digits folded in (arguments as
// ks_moddown_mac)
template <int PARTS>
void moddown_mac(Context& c, int level, int n, const KsItem* items, const u64* D, long long dstride, u64* AP, u64* T,
                 bool montgomery, hipStream_t s, int first, int period);

}  // namespace mi
