// Launchers of the z pass (cfg_z.hip), used by the nonlinear term.
#pragma once

#include "cfg_kernels.hpp"

namespace cfg {

size_t lds_budget();

// Whether a form's wavefront z pass runs a component per wavefront (k_zsplit) or
// all three in one (k_zwave). The forms with gradients, always: a wavefront then
// holds a third of the values and runs 4 (convection 3) transforms in a row instead
// of 11 (8), so twice as many fit a SIMD. us per launch, one wavefront -> three:
// skew-symmetric 32^3 11.1 -> 6.5, 64^3 14.0 -> 11.2, 96^3 38.8 -> 33.6, 128^3 66.7 ->
// 63.7, 192x97x192 163 -> 130, 24 of 32^3 27.4 -> 22.4, 24 of 48^3 73 -> 67, 16 of
// 64^3 100 -> 96; convection 24 of 32^3 22.0 -> 18.8, 96^3 29.6 -> 25.6, 128^3 49.3 ->
// 48.0, 192x97x192 94 -> 75. The rotational and the divergence form have few
// transforms to share out (the divergence form one more than alone): rotational
// 16x33x32 4.5 -> 3.7, 32^3 5.9 -> 4.5, 24 of them 13.9 -> 14.1, but 16 of 48^3 20.7
// -> 23.3, 16 of 64^3 43 -> 46, 192x129x192 62 -> 68; divergence 16 of 24x33x24 8.9 ->
// 8.6, but 24 of 32^3 13.1 -> 16.6, 16 of 64^3 45 -> 83. The rule looks at the grid
// alone: a member's result must not depend on which instance its batch runs.
constexpr bool zsplit(int method, int nz) {
    return method == NL_CONV || method == NL_SKEW || nz <= (method == NL_ROT ? 32 : 24);
}
// Three steps per transform (ZW3) at Nz = 72 and from 96 on. What bounds the z
// pass there is how few wavefronts a SIMD holds: with 6 physical values per lane
// instead of 8 to 16 and transforms of at most 9 values, 2 or 3 of them fit the
// registers where 1 did (skew-symmetric 96: 341 -> 162 registers, rotational
// 192: 297 -> 131), at the price of a second transpose through LDS. us per
// launch, two steps -> three: one 96^3 skew-symmetric field 59 -> 44, 128^3
// convection 92 -> 70, rotational 49 -> 35, 192x129x192 rotational 95 -> 76,
// 256x33x256 52 -> 48, 64x49x162 skew-symmetric 61 -> 32, 8 members of 32x49x72
// 72 -> 53; with a component per wavefront (k_zsplit) 96^3 skew-symmetric 37 -> 34,
// 128^3 convection 62 -> 52. At 48 and 64, where 2 wavefronts fit anyway, the second transpose
// costs more than it gives in a batch (16 of 64^3 113 -> 127, 24 of 48^3 82 -> 88).
constexpr bool zwave_three(int nz) { return nz == 72 || nz >= 96; }
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
