// transfer.hip -- particle records between the caller's host array and the
// device copy (vpm_set_particles, vpm_add_particles, vpm_get_particles).
//
// The caller's array is pageable, so the runtime copies through a staging
// buffer of its own on one thread, and a row range was then scattered on one
// more pass: 28 ms for the 33 rows of 262,144 particles (69 MB), 70 ms for the
// 15 rows of 2^20 -- for kernels that run in 1.5 and 350 ms.  Here a transfer
// runs through a ring of kSlots pinned pieces of 1-4 MiB: the device copies
// (or gathers rows) into one piece while host threads move another.  Row
// ranges need no device buffer (the gather writes the pinned piece itself).
//
// Pinning a ring takes 0.2-2 ms, so rings outlive a transfer: a transfer takes
// an idle one and gives it back when its stream has passed it.  At most
// kIdleRings (12 MiB each) are kept, and none once the last field is gone.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "host_team.h"
#include "vpm_internal.h"

namespace vpm {

constexpr int kSlots = 3;
// Uploads through the ring: small ones (the runtime takes 167 us for 368 KB,
// the ring 25) and large ones (96 MB 5.2 -> 2.7 ms with four threads); between
// them the runtime's own staging is as fast, and needs no ring.
constexpr size_t kSmallUpload = (size_t)2 << 20, kLargeUpload = (size_t)32 << 20;

// Bytes of a ring piece for a transfer.
static size_t piece_bytes(size_t total)
{
    const size_t mib = (size_t)1 << 20;
    return std::min(4 * mib, std::max(mib, total / 16));
}

// out[i][r] = P[i][row0 + r] for np records
__global__ __launch_bounds__(kBlock) void gather_rows_kernel(const double* __restrict__ P, int64_t np, int row0,
                                                             int nr, double* __restrict__ out)
{
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= np * nr) return;
    const int64_t i = k / nr;
    const int r = (int)(k - i * nr);
    out[k] = P[i * NF + row0 + r];
}

namespace {

constexpr size_t kIdleRings = 4;
std::mutex g_ring_mu;
std::vector<DevBuf> g_idle;      // guarded by g_ring_mu
int64_t g_fields = 0;            // live fields

// A ring for one transfer; nothing of it is in flight when it is destroyed.
struct Ring {
    DevBuf b;
    ~Ring()
    {
        if (!b.p) return;
        {
            std::lock_guard<std::mutex> lk(g_ring_mu);
            if (g_fields > 0 && g_idle.size() < g_idle.capacity()) {
                g_idle.push_back(b);
                return;
            }
        }
        (void)hipHostFree(b.p);
    }
    int take(size_t bytes)
    {
        {
            std::lock_guard<std::mutex> lk(g_ring_mu);
            for (DevBuf& i : g_idle) {
                if (i.bytes < bytes) continue;
                b = i;
                i = g_idle.back();
                g_idle.pop_back();
                return VPM_OK;
            }
            if (g_idle.size() == kIdleRings) {   // all too small: the new one takes a place
                b = g_idle.back();
                g_idle.pop_back();
            }
        }
        if (b.p) {
            (void)hipHostFree(b.p);
            b = DevBuf();
        }
        const size_t want = std::max(bytes, (size_t)kSlots << 20);
        const hipError_t e = hipHostMalloc(&b.p, want, hipHostMallocPortable);
        if (e != hipSuccess) {
            b.p = nullptr;
            return hip_fail(e, "hipHostMalloc(transfer ring)");
        }
        b.bytes = want;
        return VPM_OK;
    }
};

// Events of the pieces in flight, for one call.  With a release to the system:
// the gather kernel writes pinned pieces that need not be coherent, and the
// host reads one after its event, with later pieces still in flight (no wait
// for the stream between).
struct Events {
    hipEvent_t ev[kSlots] = {};
    ~Events()
    {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    }
    int make(int n)
    {
        for (int s = 0; s < n; ++s) {
            const hipError_t e = hipEventCreateWithFlags(&ev[s], hipEventDisableTiming | hipEventReleaseToSystem);
            if (e != hipSuccess) return hip_fail(e, "hipEventCreate");
        }
        return VPM_OK;
    }
};

// [a, b) of worker w of n over `count` items
void share(int64_t count, int w, int n, int64_t& a, int64_t& b)
{
    a = count * w / n;
    b = count * (w + 1) / n;
}

}  // namespace

int transfer_field(int change)
{
    std::vector<DevBuf> freed;
    try {
        std::lock_guard<std::mutex> lk(g_ring_mu);
        if (change > 0) g_idle.reserve(kIdleRings);
        g_fields += change;
        if (g_fields == 0) freed.swap(g_idle);
    } catch (const std::exception&) {
        return fail(VPM_ENOMEM, "transfer rings");
    }
    for (DevBuf& b : freed) (void)hipHostFree(b.p);
    return VPM_OK;
}

int check_records(const double* p, int64_t np)
{
    HostTeam team(team_size(sizeof(double) * NF * (size_t)np));
    // the first bad particle of each worker's share (0: none), lowest first
    int64_t bad[8];
    for (int64_t& b : bad) b = -1;
    team.run([&](int w, int n) {
        int64_t a, e;
        share(np, w, n, a, e);
        for (int64_t i = a; i < e; ++i) {
            const double* r = p + i * NF;
            bool ok = r[RSIG] > 0;
            for (int k = 0; k < 7; ++k) ok = ok && std::isfinite(r[k]);
            if (!ok) { bad[w] = i; return; }
        }
    });
    for (const int64_t i : bad) {
        if (i < 0) continue;
        for (int k = 0; k < 7; ++k)
            if (!std::isfinite(p[i * NF + k]))
                return fail(VPM_EINVAL, "non-finite X/Gamma/sigma at particle " + std::to_string(i));
        return fail(VPM_EINVAL, "sigma <= 0 at particle " + std::to_string(i));
    }
    return VPM_OK;
}

int upload_records(vpm_field f, const double* src, int64_t first, int64_t np)
{
    const size_t rec = sizeof(double) * NF;
    const size_t total = rec * (size_t)np;
    if (total > kSmallUpload && total < kLargeUpload) {
        hipError_t e = hipMemcpyAsync(f->P + first * NF, src, total, hipMemcpyHostToDevice, f->stream);
        const hipError_t w = hipStreamSynchronize(f->stream);
        if (e == hipSuccess) e = w;
        return e == hipSuccess ? VPM_OK : hip_fail(e, "hipMemcpyAsync(H2D)");
    }
    const int64_t per = std::min<int64_t>(np, (int64_t)(piece_bytes(rec * (size_t)np) / rec));
    const int64_t pieces = (np + per - 1) / per;
    const int slots = (int)std::min<int64_t>(kSlots, pieces);
    Ring ring;
    if (int rc = ring.take((size_t)slots * per * rec)) return rc;
    Events ev;
    if (int rc = ev.make(pieces > kSlots ? slots : 0)) return rc;
    HostTeam team(team_size(rec * (size_t)np));
    int rc = VPM_OK;
    for (int64_t k = 0; k < pieces && !rc; ++k) {
        const int s = (int)(k % slots);
        const int64_t a = k * per, n = std::min(per, np - a);
        char* slot = (char*)ring.b.p + (size_t)s * per * rec;
        hipError_t e = k >= slots ? hipEventSynchronize(ev.ev[s]) : hipSuccess;
        if (e != hipSuccess) { rc = hip_fail(e, "hipEventSynchronize"); break; }
        team.run([&](int w, int m) {
            int64_t b, c;
            share(n, w, m, b, c);
            std::memcpy(slot + b * rec, src + (a + b) * NF, rec * (size_t)(c - b));
        });
        e = hipMemcpyAsync(f->P + (first + a) * NF, slot, rec * (size_t)n, hipMemcpyHostToDevice, f->stream);
        if (e == hipSuccess && ev.ev[s]) e = hipEventRecord(ev.ev[s], f->stream);
        if (e != hipSuccess) rc = hip_fail(e, "hipMemcpyAsync(H2D)");
    }
    // the ring is free again when the call returns, also on failure
    const hipError_t e = hipStreamSynchronize(f->stream);
    return rc ? rc : e == hipSuccess ? VPM_OK : hip_fail(e, "hipStreamSynchronize");
}

int download_rows(vpm_field f, double* dst, int64_t np, int row0, int row1)
{
    const int nr = row1 - row0;
    const size_t rec = sizeof(double) * (size_t)nr;
    const int64_t per = std::min<int64_t>(np, (int64_t)(piece_bytes(rec * (size_t)np) / rec));
    const int64_t pieces = (np + per - 1) / per;
    const int slots = (int)std::min<int64_t>(kSlots, pieces);
    Ring ring;
    if (int rc = ring.take((size_t)slots * per * rec)) return rc;
    Events ev;
    if (int rc = ev.make(pieces > 1 ? slots : 0)) return rc;
    const auto issue = [&](int64_t k) -> int {
        const int s = (int)(k % slots);
        const int64_t a = k * per, n = std::min(per, np - a);
        double* slot = (double*)((char*)ring.b.p + (size_t)s * per * rec);
        hipError_t e;
        if (nr == NF) {
            e = hipMemcpyAsync(slot, f->P + a * NF, rec * (size_t)n, hipMemcpyDeviceToHost, f->stream);
        } else {
            hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)((n * nr + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                               f->stream, f->P + a * NF, n, row0, nr, slot);
            e = hipGetLastError();
        }
        if (e == hipSuccess && ev.ev[s]) e = hipEventRecord(ev.ev[s], f->stream);
        return e == hipSuccess ? VPM_OK : hip_fail(e, "particle download");
    };
    HostTeam team(team_size(rec * (size_t)np));
    int rc = VPM_OK;
    int64_t issued = 0;
    for (int64_t k = 0; k < pieces && !rc; ++k) {
        while (issued < pieces && issued < k + slots && !rc) rc = issue(issued++);
        if (rc) break;
        const int s = (int)(k % slots);
        const hipError_t e = ev.ev[s] ? hipEventSynchronize(ev.ev[s]) : hipStreamSynchronize(f->stream);
        if (e != hipSuccess) { rc = hip_fail(e, "particle download"); break; }
        const int64_t a = k * per, n = std::min(per, np - a);
        const char* slot = (const char*)ring.b.p + (size_t)s * per * rec;
        team.run([&](int w, int m) {
            int64_t b, c;
            share(n, w, m, b, c);
            if (nr == NF) {
                std::memcpy(dst + (a + b) * NF, slot + b * rec, rec * (size_t)(c - b));
            } else {
                for (int64_t i = b; i < c; ++i) std::memcpy(dst + (a + i) * NF + row0, slot + i * rec, rec);
            }
        });
    }
    if (rc) (void)hipStreamSynchronize(f->stream);   // no launch still writes the ring
    return rc;
}

}  // namespace vpm
