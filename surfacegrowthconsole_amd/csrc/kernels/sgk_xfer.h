// sgk_xfer.h - state transfer between host arrays in the reference layouts (positions x,y,z,E;
// velocities and accelerations x,y,z per atom) and the device's storage (sgk_xfer.hip).
//
// A pageable hipMemcpy costs ~130 us from 0.3 MB on and moves 88 MB (1.1 M atoms) in 5-9 ms, and the
// layouts were converted on the host, one array after another.  Here one kernel per piece converts
// between the device arrays and a pinned slot of the context, and the kernel of one slot runs while
// the host copies the other, with several host threads where the state is large (the page faults of a
// fresh array are shared then too).  No device memory is needed.  Download of everything as doubles:
// 68 -> 20 us at 1,161 atoms, 328 -> 135 at 44,353, 15.4 -> 2.8 ms at 1.1 M; upload 65 -> 19 us,
// 216 -> 139, 5.3 -> 2.8 ms.  A device stage with copy-engine transfers took 39, 188 and 3,093 us and its
// allocation made a context's first download 1 ms longer.  Slots of
// 256 KiB, 512 KiB and 1 MiB: 177, 136 and 145 us at 44,353 atoms, 3.8, 2.9 and 2.4 ms at 1.1 M; a
// context's first transfers (pages pinned and touched) 0.3, 0.5 and 1.7 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace sgk {

constexpr int kXferThreads = 8;                     // host threads of a large transfer
constexpr size_t kXferSlot = (size_t)512 << 10;     // most bytes of a pinned slot; two per thread
constexpr size_t kXferWhole = (size_t)256 << 10;    // below, one piece for everything
// Transfers from here on use kXferThreads threads: starting them costs ~70 us, more than the rest of
// a 4 MB transfer to a warm array (257 against 188 us) and less than they save at 8 MB (510 against 910 us).
constexpr size_t kXferLarge = (size_t)8 << 20;

// Pinned slots, grown on demand, owned by a context or a batch (one transfer at a time per owner, as
// every call on it).
struct HostStage {
    char *pin = nullptr;
    size_t bytes = 0;
    hipEvent_t ev[2 * kXferThreads] = {};
};
void stage_free(HostStage &st);

// One host array of doubles or floats and the device array it mirrors.
enum class XferLayout : int {
    plain,   // value j
    blocks,  // x, y and z of each atom on the host, blocks of all x, y and z on the device
    energy,  // w of the j-th position
};
struct XferArray {
    void *host;
    const void *dev;   // written by a transfer to the device
    size_t count;      // values on the host (3n for blocks)
    XferLayout layout;
    bool wide;         // stored as doubles on the device, else floats
};
// H: the host's type.  The n arrays (at most 3) move after what stream s holds and before what
// follows on it; on return the host's are complete, or no longer needed.
template <class H>
hipError_t xfer_to_host(HostStage &st, int device, hipStream_t s, const XferArray *arrays, int n);
// The state of n atoms, any of the host arrays null: r 4n, v 3n, a 3n.
template <class H>
hipError_t state_to_host(HostStage &st, int device, hipStream_t s, size_t n, bool wide, const void *pos, const void *vel,
                         const void *acc, H *r, H *v, H *a);
template <class H>
hipError_t state_to_device(HostStage &st, int device, hipStream_t s, size_t n, bool wide, const H *r, const H *v,
                           const H *a, void *pos, void *vel, void *acc);

}  // namespace sgk
