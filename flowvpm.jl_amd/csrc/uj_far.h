// uj_far.h -- F32C all-pairs U/J with the far field on the matrix cores
// (uj_far.hip), as launch_uj (p2p_uj.hip) uses it.
#pragma once
#include "vpm_internal.h"

namespace vpm {

// Fewest particles of a field whose time steps take the far kernel.
constexpr int64_t kFarStepMin = 1 << 16;

// Whether an all-pairs launch is split at all.
bool far_applies(int kernel, int precision, int64_t nt, int64_t ns);
// Partial sums [k.far + k.rest][kAccF32][nt] of sources [0, ns) of S on
// targets [t0, t0 + nt) of T.
int launch_uj_far(hipStream_t stream, const Staged& T, int64_t t0, int64_t nt, const Staged& S, int64_t ns, int kernel,
                  const FarSplit& k, void* scratch, double* part);

}  // namespace vpm
