// What the two compact-function kernels share.
#pragma once

#include "kernels.hpp"

namespace nnpx {

enum CompMode { CM_PLAIN = 0, CM_VALUES = 1, CM_FORCE = 2, CM_TANGENT = 3 };

// Outputs of the mixed modes.
struct CompMix {
    double* G;        // [N*ldG] scaled values (values mode)
    float* Gin;       // [N*ldK] their FP32 copy, the network input
    int ldG, ldK;
    const float* fw;  // [N*ldG] dE/dG times the scaling factor (force mode)
    double* F;        // forces (force mode)
    int push;         // keep contributions to the atom's own images
    const double* u;  // [3N] field of the tangent mode (its output goes to G)
    const double* fw64;  // [N*ldG] FP64 weights of the FP64 force mode (plain form)
};

// Radial groups and factored angular groups of every atom in one of the modes
// (values, force, tangent), FP32 or FP64 terms.
template <typename T>
void launch_sfcomp_factored(const ModelT* m, const ModelT& hm, const SysView& s, const CompMix& c, CompMode mode,
                            int capL, hipStream_t stream);
// Whether that kernel can stage capL neighbours.
template <typename T>
bool sfcomp_factored_fits(CompMode mode, int capL);

}  // namespace nnpx
