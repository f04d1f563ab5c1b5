// Device side of the serial coordinate-descent deconvolver (FastSerialCD.cs)
// and of the PSF correlation (PaddedConvolver.cs, Common.cs PSF helpers).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace p9idg {
namespace cd {

constexpr int kTile = 32;  // edge of the argmax tiles (pixels)

// A candidate update as an ordered word (kernels_cd.hip); 0: none.
using Key = unsigned long long;

// Results of the deconvolver's kernels.
struct State {
    int32_t done;       // no further updates
    int32_t converged;  // the last selected |diff| was below epsilon
    int32_t updates;    // pixels changed by the launch
    int32_t stalled;    // the workgroups were not all resident (1: nothing was changed)
    float absmax;       // GetAbsMaxDiff
    int32_t pad[3];
};

// All tiles of the table for lambda / alpha.
hipError_t launch_tiles_all(const float* x, const float* g, const float* amap, int H, int W, float lambda,
                            float alpha, Key* tiles, hipStream_t st);
// GetAbsMaxDiff: the best |diff| of the tile table into state->absmax.
hipError_t launch_absmax(const Key* tiles, int ntiles, State* state, hipStream_t st);

// The descent's workgroups: OH x OW of them on the current device, `local`
// tiles each at most.
struct DescentShape {
    int OH = 0, OW = 0, local = 0;
};
hipError_t descent_shape(int H, int W, int p2h, int p2w, DescentShape* shape);
size_t descent_slots(const DescentShape& shape);  // words
// kResident: gradients in LDS, one workgroup per CU; kShared: gradients in
// memory, beside other kernels' workgroups; kSingle: one workgroup, which waits
// for nobody.
enum DescentForm { kResident, kShared, kSingle };
DescentForm descent_form(const DescentShape& shape);  // the fastest that fits
// Up to `limit` (> 0) iterations on x and g.  tiles: max(OH OW local, all tiles)
// words.
hipError_t launch_descent(float* x, float* g, const float* amap, const float* psf2, int p2h, int p2w, int H, int W,
                          const DescentShape& shape, DescentForm form, float lambda, float alpha, float epsilon, int limit,
                          Key* slots, Key* tiles, State* state, hipStream_t st);

// PaddedConvolver / CalcPaddedFourierCorrelation pieces (complex double
// buffers of N0 x N1).
hipError_t launch_place_correlation(const float* psf, int ph, int pw, int ypad, int xpad, int N0, int N1,
                                    double2* buf, hipStream_t st);
hipError_t launch_place_centered(const float* psf, int ph, int pw, int N0, int N1, double2* buf,
                                 hipStream_t st);
hipError_t launch_insert_image(const float* img, int H, int W, int yh, int xh, int N0, int N1, double2* buf,
                               hipStream_t st);
hipError_t launch_multiply(double2* buf, const double2* kernel, size_t n, hipStream_t st);
// out[y][x] = (float)(Re buf[y + yh][x + xh] / norm)
hipError_t launch_extract(const double2* buf, int N1, int yh, int xh, double norm, int H, int W, float* out,
                          hipStream_t st);
// Common.cs:48-126 per pixel from the prefix sums of psf^2
hipError_t launch_amap(const double* scan, int ph, int pw, int H, int W, float* amap, hipStream_t st);
// max(0, max_i v[i]) into *out (Residuals.GetMax)
hipError_t launch_get_max(const float* v, size_t n, float* out, hipStream_t st);

}  // namespace cd
}  // namespace p9idg
