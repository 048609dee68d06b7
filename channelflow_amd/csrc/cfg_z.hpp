// Launchers of the z pass (cfg_z.hip), used by the nonlinear term.
#pragma once

#include "cfg_kernels.hpp"

namespace cfg {

size_t lds_budget();

// real physical lines per (y, x) line the LDS z-pass of a form keeps
int zpass_nphys(int method);
// largest LDS z-pass lines per block that fit the LDS budget
int zpass_xb_max(const Geom& g, int nphys);
// z pass of n members (strides sx in double2): fields of xp to fields of zo
void launch_z_any(int method, const Geom& g, const FFTPlan& pz, int n, const NLMember* tab, int want_g,
                  const double2* xp, double2* zo, long sx, const NLTune& tn, hipStream_t st);
// partial maxima of the CFL factor, per member as many as returned
int launch_zcfl(const Geom& g, const FFTPlan& pz, int n, const NLMember* tab, const double2* xp, long sx, double* part,
                hipStream_t st);
// the maximum of each member's nb partial maxima
void launch_cfl_reduce(int n, int nb, const double* part, double* out, hipStream_t st);

}  // namespace cfg
