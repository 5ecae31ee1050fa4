// bf_ring.h -- the unrolled kernels of the canonical ring template for one
// image or a device tile list (tile_ring in bf_tile.h), and their launch.
// Each (mode, tile, halo) is instantiated in one of the bf_ring_*.hip files,
// so that they compile in parallel.  Not a public header.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "bf_internal.h"
#include "bf_tile.h"

namespace bfimpl {

// One image, static grid-stride over its tiles (or over the tiles of a
// device list, whose length is read on the device); job.rowg holds the
// per-q weights of the canonical template and job.nrows how many of them the
// LDS table holds.
// (Cutting the last round's tiles into four-group quarters shared by all
// workgroups measured slower, 360 against 344 us at r = 7 on 3800 x 3600: a
// SIMD needs its four waves to cover the gathers' latency.  Equal runs of
// groups down the columns took 366 us, and 7.95 against 7.67 ms at r = 15 on
// 8192^2: every workgroup then stages rows of its own part of the image.)
template <int MODE, int TW, int TGY, int HALO>
__global__ void __launch_bounds__(TW * TGY)
bf_ring_kernel(DevJob job, int ntiles, const int32_t *list, const int32_t *list_count)
{
    using G = Geo<TW, TGY, HALO>;
    const int tid = threadIdx.x;
    const int lx = tid % TW, gy = tid / TW;
    build_lut<G::NT>(job, kTileOff + (uint32_t)G::TILE_BYTES, tid);
    const int n = list ? *as_const(list_count) : ntiles;
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const int tile = list ? as_const(list)[i] : i;
        const int ty = tile / job.tiles_x;
        const int X0 = (tile - ty * job.tiles_x) * TW;
        const int Y0 = ty * G::TH;
        __syncthreads();                      // table built / previous tile consumed
        load_tile<TW, TGY, HALO>(job, X0, Y0, tid);
        __syncthreads();
        tile_ring<MODE, TW, TGY, HALO, halo_min_radius(HALO), ring_group<MODE, HALO, false>()>(job, X0, Y0, lx, gy);
    }
}

template <int MODE, int TW, int TGY, int HALO>
int launch_ring_one(const DevJob &job, int ntiles, const int32_t *list, const int32_t *count,
                    hipStream_t s)
{
    using G = Geo<TW, TGY, HALO>;
    constexpr auto kern = bf_ring_kernel<MODE, TW, TGY, HALO>;
    const size_t lds = kTileOff + (size_t)G::TILE_BYTES + (size_t)job.lut_rows * 1024;
    BF_HIP(allow_full_lds<kern>());
    const int res = resident_groups(reinterpret_cast<const void *>(kern), G::NT, lds);
    if (res < 0) return hip_fail(hipGetLastError(), "occupancy query");
    if (res < 1) {
        set_error("ring kernel does not fit on a CU");
        return kInvalidData;
    }
    const int grid = std::min(ntiles, res);   // with a list, ntiles = its maximum length
    if (grid < 1) return kOk;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(G::NT), lds, s, job, ntiles, list, count);
    BF_HIP(hipGetLastError());
    return kOk;
}

#define BF_RING_KERNEL(X, MODE, TW, TGY, HALO)                                                 \
    X template int launch_ring_one<MODE, TW, TGY, HALO>(const DevJob &, int, const int32_t *, \
                                                        const int32_t *, hipStream_t);
// The instances: 64 x 16 tiles to r = 8, 64 x 32 tiles (REF to r = 16), 64 x
// 64 tiles from r = 9.
#define BF_RING_SMALL(X, MODE)           \
    BF_RING_KERNEL(X, MODE, 64, 4, 4)    \
    BF_RING_KERNEL(X, MODE, 64, 4, 8)    \
    BF_RING_KERNEL(X, MODE, 64, 8, 4)    \
    BF_RING_KERNEL(X, MODE, 64, 8, 8)    \
    BF_RING_KERNEL(X, MODE, 64, 8, 12)
#define BF_RING_MID(X, MODE)             \
    BF_RING_KERNEL(X, MODE, 64, 16, 12)  \
    BF_RING_KERNEL(X, MODE, 64, 16, 16)
#define BF_RING_LARGE(X, MODE)           \
    BF_RING_KERNEL(X, MODE, 64, 8, 16)   \
    BF_RING_KERNEL(X, MODE, 64, 16, 20)
#define BF_RING_STD_LARGE(X) BF_RING_KERNEL(X, 1, 64, 8, 20)

}  // namespace bfimpl
