// uj_split.h -- how launches are split over source splits, and what their
// workspace takes.  Host only, no device code.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "../../include/flowvpm_hip.h"

namespace vpm {

constexpr int kBlock = 256;      // threads per block (4 waves of 64)
constexpr int kTile = 256;       // sources per LDS tile
constexpr int kAccF32 = 14;      // U'(3) W'(3) Jhv(8) per target, F32C path
constexpr int kAccF64 = 12;      // U(3) J(9) per target, F64 path

// Workspace for K splits by take(K), with half of them where memory does not
// hold it (VPM_ENOMEM), down to one: fewer splits run longer, and the sums
// group otherwise, but a field that fits in memory is evaluated.
template <class Take>
int fit_splits(int64_t& K, Take&& take)
{
    for (;;) {
        const int rc = take(K);
        if (rc != VPM_ENOMEM || K <= 1) return rc;
        K = (K + 1) / 2;
    }
}

// ---- the far kernel and its rest kernel (uj_far.hip) ----
// Source splits of the two kernels of a launch.
struct FarSplit {
    int64_t far = 1, chunk = 1;   // far kernel: splits, tiles per split
    int64_t rest = 1;             // rest kernel: splits (every rest-th tile)
};

// Blocks of a launch.  The far kernel's blocks do equal work per tile; 2,048
// or 8,192 of them measure the same at N = 65,536, and fewer splits leave
// fewer partial sums.  The rest kernel's work per wave is uneven (a wave whose
// targets are scattered reaches most sources), so it has at least 16 splits:
// 352 ms at 2^20 with 16 or more, 358 with 8, 401 with 2.
constexpr int64_t kFarBlocks = 2048;
constexpr int64_t kRestBlocks = 4096;
constexpr int64_t kRestMin = 16;

// Targets per launch: the words of one launch stay within 256 MiB.
inline int64_t far_batch(int64_t nt, int64_t ns)
{
    const int64_t ntile = (ns + kTile - 1) / kTile;
    const int64_t most = std::max<int64_t>(1, ((int64_t)64 << 20) / ntile) * kBlock;
    return std::min(nt, most);
}

inline int64_t far_up256(int64_t b) { return (b + 255) & ~(int64_t)255; }

// Scratch of one launch (boxes and words).
inline size_t far_scratch_bytes(int64_t nt, int64_t ns)
{
    const int64_t nwave = (nt + 63) / 64, ngroup = (ns + 63) / 64;
    const int64_t nblk = (nt + kBlock - 1) / kBlock, ntile = (ns + kTile - 1) / kTile;
    return (size_t)(far_up256(64 * nwave) + far_up256(64 * ngroup) + far_up256(4 * nblk * ntile));
}

// Partial sums of one launch over nt targets.
inline size_t far_part_bytes(int64_t nt, const FarSplit& k)
{
    return sizeof(double) * kAccF32 * (size_t)(k.far + k.rest) * (size_t)nt;
}

// kmax > 0 caps each kernel's splits.
inline FarSplit far_split(int64_t nt, int64_t ns, int64_t kmax)
{
    const int64_t nblk = (nt + kBlock - 1) / kBlock, ntile = (ns + kTile - 1) / kTile;
    const auto cap = [&](int64_t K) {
        K = std::max<int64_t>(1, K);
        if (kmax > 0) K = std::min(K, kmax);
        return std::min(K, ntile);
    };
    FarSplit k;
    k.far = cap(kFarBlocks / nblk);
    k.chunk = (ntile + k.far - 1) / k.far;
    k.far = (ntile + k.chunk - 1) / k.chunk;
    k.rest = cap(std::max<int64_t>(kRestMin, kRestBlocks / nblk));
    return k;
}

// The splits of a launch whose partial sums take(bytes) finds memory for.
template <class Take>
int fit_far_split(int64_t nt, int64_t ns, int64_t kmax, FarSplit& k, Take&& take)
{
    k = far_split(nt, ns, kmax);
    int64_t most = std::max(k.far, k.rest);
    return fit_splits(most, [&](int64_t m) {
        k = far_split(nt, ns, m);
        return take(far_part_bytes(nt, k));
    });
}

}  // namespace vpm
