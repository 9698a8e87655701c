// Few-token product instantiations for IQ2_XXS, IQ2_XS; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_IQ2_XXS>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ2_XXS>(bool, int, int, int);
template hipError_t skinny_dispatch<T_IQ2_XS>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ2_XS>(bool, int, int, int);
}  // namespace qm
