// uj_far.h -- F32C all-pairs U/J with the far field on the matrix cores
// (uj_far.hip), as launch_uj (p2p_uj.hip) uses it.
#pragma once
#include "vpm_internal.h"

namespace vpm {

// Fewest particles of a field whose time steps take the far kernel (the line
// that keeps a step's results what they are: uj_direct_locked in vpm_abi.hip;
// it would pay from 18,000: steps of the cloud, the jet, the leapfrog rings and
// a thin ring 2.03 / 1.84 / 2.03 / 1.76 -> 1.77 / 1.58 / 1.84 / 1.53 ms at 20,000).
constexpr int64_t kFarStepMin = 1 << 16;

// Whether an all-pairs launch is split at all.
bool far_applies(int kernel, int precision, int64_t nt, int64_t ns);
// Partial sums [k.far + k.rest][kAccF32][nt] of sources [0, ns) of S on
// targets [t0, t0 + nt) of T.
int launch_uj_far(hipStream_t stream, const Staged& T, int64_t t0, int64_t nt, const Staged& S, int64_t ns, int kernel,
                  const FarSplit& k, void* scratch, double* part);

}  // namespace vpm
