// The z pass of the rotational form.
#include <hip/hip_runtime.h>

#include "cfg_zpass.hpp"

namespace cfg {

template void launch_z<NL_ROT>(const Geom&, const FFTPlan&, int, const NLMember*, int, const double2*, double2*,
                               long, const NLTune&, hipStream_t);

}  // namespace cfg
