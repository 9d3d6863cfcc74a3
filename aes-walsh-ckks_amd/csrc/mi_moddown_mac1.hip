#include "mi_moddown_mac.hpp"

namespace mi {
template void moddown_mac<1>(Context&, int, int, const KsItem*, const u64*, long long, u64*, u64*, bool, hipStream_t,
                             int, int);
}  // namespace mi
