// The z pass of the convection form.
#include <hip/hip_runtime.h>

#include "cfg_zpass.hpp"

namespace cfg {

template void launch_z<NL_CONV>(const Geom&, const FFTPlan&, int, const NLMember*, int, const double2*, double2*,
                               long, const NLTune&, hipStream_t);

}  // namespace cfg
