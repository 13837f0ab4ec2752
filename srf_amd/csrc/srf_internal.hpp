// srf_internal.hpp -- helpers shared by the translation units of libsrf_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "srf_hip.h"

namespace srf {

// Status of the launches just issued (hipGetLastError clears the sticky error
// of a failed launch, so each entry point reports its own).
inline int launch_status()
{
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? SRF_OK : SRF_ERR_LAUNCH;
}

// dst[i] = v for i < n.  A kernel, not hipMemsetAsync, so the call may be
// captured into a HIP graph and replayed.
int fill_f32(float *dst, float v, int64_t n, hipStream_t s);

// Device memory for plans and scratch (srf_pool.hip).  pool_get: at least `bytes`
// on the current device, for use in stream order on s (nullptr: none left).
// pool_put: given back once the work queued on s so far is done (idle: nothing
// uses it any more; scratch: not a plan's, of which the pool keeps less).  Not for
// a stream that is being captured.  Neither throws.
void *pool_get(size_t bytes, hipStream_t s);
void pool_put(void *p, hipStream_t s, bool idle = false, bool scratch = false);

// True on a stream that is being captured (no scratch can be taken for it then),
// or whose state cannot be told.
inline bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return st != hipStreamCaptureStatusNone;
}

struct LaunchGeom;
// Validates a grid (and TOF parameters) and derives the per-launch constants.
int make_geom(const srf_grid_t &g, const srf_tof_t *tof, LaunchGeom &G);

// Backprojection of one list through a plan of its own (srf_tiled.hip); anything but
// SRF_OK: nothing was added to the image.  SRF_ERR_WORKSPACE: the list has more segments
// than a call may take scratch for, `fit` of its events would do.  Synchronises s.
int backproject_binned(const float *lors, int64_t n, int64_t lor_stride, const float *tof_values, int64_t tof_stride,
                       const float *values, const float *y, const float *p, int kind, float eps, srf_grid_t grid,
                       const srf_tof_t *tof, srf_bp_mode_t mode, int accumulate, float *image, hipStream_t s, int64_t &fit);

}  // namespace srf
