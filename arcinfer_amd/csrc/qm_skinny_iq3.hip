// Few-token product instantiations for IQ3_S, IQ3_XXS; the kernels are in qm_skinny_impl.h.
#include "qm_skinny_impl.h"

namespace qm {
template hipError_t skinny_dispatch<T_IQ3_S>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ3_S>(bool, int, int, int);
template hipError_t skinny_dispatch<T_IQ3_XXS>(const SkinnyArgs&, hipStream_t);
template bool skinny_takes<T_IQ3_XXS>(bool, int, int, int);
}  // namespace qm
