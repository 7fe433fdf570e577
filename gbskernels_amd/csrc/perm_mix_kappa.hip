// perm_mix_kappa.hip -- the multi-size permanent launch, kappa tier.
#include "perm_mix_impl.hpp"

namespace gbsk {
template void perm_mix_launch<PERM_KAPPA, false>(const PermMix&, hipStream_t);
template void perm_mix_launch<PERM_KAPPA, true>(const PermMix&, hipStream_t);
}
