// aux_launch.hpp -- host launchers of the auxiliary kernels (aux.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "physics.hpp"

namespace glm {

constexpr size_t DIAG_CELLS_PER_BLOCK = 16384;

// Workgroups of a whole-grid max reduction: two cells a lane until 1024 workgroups (4 per CU), then more
// cells a lane, since every workgroup ends with an atomic on the same address.  64^3 FP64: 4.5 us with
// 512 workgroups, 6.5 with 128; 128^3: 24 us with 1024, 40 with 2048.
inline unsigned red_blocks(size_t n)
{
    const size_t g = (n + 511) / 512;
    return (unsigned)(g < 1024 ? g : 1024);
}

hipError_t launch_clear_u64(unsigned long long* p, int n, hipStream_t st);
// *host = *slot (host: device-mapped host memory), then *slot = 0 when clear.
hipError_t launch_publish_u64(unsigned long long* slot, unsigned long long* host, bool clear, hipStream_t st);
template <typename T>
hipError_t launch_ctot(Ptr9<const T> q9dev, size_t n, const Phys<T>& s, unsigned long long* out, hipStream_t st,
                       bool fast = false);
size_t diag_nparts(size_t n);
size_t diag_part_bytes();
template <typename T>
hipError_t launch_diag(Ptr9<const T> q9dev, int nx, int ny, int nz, double dx, double smallr, void* parts,
                       double* out, hipStream_t st);
template <typename T>
hipError_t launch_ic(Ptr9<T> q9dev, int nx, int ny, int nz, int kind, const double* args, hipStream_t st);

}  // namespace glm
