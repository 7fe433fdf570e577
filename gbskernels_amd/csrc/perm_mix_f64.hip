// perm_mix_f64.hip -- the multi-size permanent launch, fp64 tier.
#include "perm_mix_impl.hpp"

namespace gbsk {
template void perm_mix_launch<PERM_FP64, false>(const PermMix&, hipStream_t);
template void perm_mix_launch<PERM_FP64, true>(const PermMix&, hipStream_t);
}
