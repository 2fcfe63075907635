// fbp.h -- standard parallel-beam geometry shared by the FBP host object and
// its kernels (kernels_fbp.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ske {

struct FbpGeom {
    int n;        // image side
    int nang;     // projection angles
    int ndet;     // detector bins
    int nt;       // ray samples per bin (= ndet)
    float delta;  // pixel pitch and bin spacing, 2/n
    float det_c;  // (ndet-1)/2
    float tmax;   // (nt-1)/2 * delta
    float pad;
};

// Tiles of the projector for S slices at a time (1 or 4): the base pixels
// [-1, n) of each axis in ntx tiles of side ts <= kPtMaxS; kw partial sums per
// (slice, angle, tile), enough for every bin that can cross a tile (ts sqrt(2)
// plus margins).
constexpr int kPtMax1 = 129, kPtMax4 = 67;
constexpr int kPtAngles = 12;  // angles per projector workgroup, at most
struct ProjTiling {
    int ntx;
    int ts;
    int kw;
};
inline ProjTiling proj_tiling(int n, int slices) {
    const int most = slices == 1 ? kPtMax1 : kPtMax4;
    ProjTiling t;
    t.ntx = (n + 1 + most - 1) / most;
    t.ts = (n + 1 + t.ntx - 1) / t.ntx;
    t.kw = (t.ts * 1415 + 999) / 1000 + 8;
    return t;
}
// Partial sums (floats) of `batch` slices projected `slices` at a time.
inline size_t proj_part_floats(int n, int nang, int batch, int slices) {
    const ProjTiling t = proj_tiling(n, slices);
    return (size_t)batch * nang * t.ntx * t.ntx * t.kw;
}
// img: batch x n x n; part: `part_floats` floats of scratch, at least
// proj_part_floats(n, nang, batch, 1); four slices at a time where it holds
// the partial sums of as many.
hipError_t launch_fbp_project(const float* img, float* part, size_t part_floats, float* sino, const float2* cs,
                              const FbpGeom& g, int batch, hipStream_t s);
hipError_t launch_fbp_filter(const float* sino, float* filt, const float* taps, const FbpGeom& g, int batch,
                             hipStream_t s);
hipError_t launch_fbp_backproject(const float* filt, float* img, const float2* cs, const FbpGeom& g, int batch,
                                  float scale, hipStream_t s);

}  // namespace ske
