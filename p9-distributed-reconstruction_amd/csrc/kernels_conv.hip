// The padded PSF correlation (PaddedConvolver.cs, Common.cs:146-160) on FP64
// line transforms in LDS.
//
// The correlation is linear, so the circular size need not be the padded size
// H + rows (W + cols) itself: n is the next even 2^a 3^b 5^c from there.  Image
// and result are real: pairs of image rows share one complex transform, the n / 2 + 1 columns
// that determine the rest are transformed, multiplied by the PSF's spectrum and
// transformed back while they are in LDS, and pairs of result rows come out of
// one complex transform.  3072^2 with a 192^2 PSF moves 0.4 GB; two 2-D library
// transforms of the complex plane with an insertion, a product and an
// extraction moved 2.4 GB in 1611 us.
#include <algorithm>

#include "device_linefft.h"

namespace p9idg {
namespace dev {

constexpr int kConv = 256;  // threads of one line

// mid[c / 2][r / 2][c & 1][r & 1]: column c of row r.  A pair of rows writes 64
// contiguous bytes per pair of columns, a column reads 32.
__device__ __forceinline__ size_t mid_at(int c, int pair, int pairs) { return ((size_t)(c >> 1) * pairs + pair) * 4 + (c & 1) * 2; }

// The blocks of an XCD (workgroups go round robin over the 8) as one range of
// neighbours, so that its L2 merges their halves of a line.
__device__ __forceinline__ int xcd_range(int blk, int n) {
    const int per = (n + 7) / 8;
    return (blk & 7) * per + (blk >> 3);
}

// Rows 2 b and 2 b + 1 of `rows` x `cols` real values, from column xoff on of a
// line of n zeros; FLIP: the image turned by 180 degrees.
template <int MAXN, bool FLIP>
__global__ __launch_bounds__(kConv) void conv_rows_kernel(const float* in, int rows, int cols, int xoff, LinePlan plan,
                                                          const double2* tw, int pairs, double2* mid) {
    __shared__ double2 line[line_slots(MAXN)];
    const int t = threadIdx.x, n = plan.n;
    const int b = xcd_range(blockIdx.x, pairs);
    if (b >= pairs) return;  // whole workgroups
    const int y0 = 2 * b, y1 = y0 + 1;
    const bool two = y1 < rows;
    for (int f = t; f < n; f += kConv) {
        const int x = f - xoff < 0 ? f - xoff + n : f - xoff;  // 0 <= xoff < n
        double2 v = make_double2(0.0, 0.0);
        if (x < cols) {
            const int at = FLIP ? cols - 1 - x : x;
            v.x = in[(size_t)(FLIP ? rows - 1 - y0 : y0) * cols + at];
            if (two) v.y = in[(size_t)(FLIP ? rows - 1 - y1 : y1) * cols + at];
        }
        line[slot(f)] = v;
    }
    __syncthreads();
    line_fft<-1, MAXN, kConv>(line, plan, tw, t);
    for (int f = t; f <= n / 2; f += kConv) {
        const double2 z = line[slot(f)], c = line[slot(f ? n - f : 0)];
        double2* o = mid + mid_at(f, b, pairs);
        o[0] = make_double2(0.5 * (z.x + c.x), 0.5 * (z.y - c.y));
        o[1] = make_double2(0.5 * (z.y + c.y), 0.5 * (c.x - z.x));
    }
}

// Column c: the rows from row yoff on of a line of n zeros.  SPECTRUM: its
// transform times `scale` to spectrum[c][f]; else its product with the spectrum,
// transformed back in place.
template <int MAXN, bool SPECTRUM>
__global__ __launch_bounds__(kConv) void conv_columns_kernel(double2* mid, int rows, int yoff, LinePlan plan,
                                                             const double2* tw, int pairs, double scale, double2* spectrum) {
    __shared__ double2 line[line_slots(MAXN)];
    const int t = threadIdx.x, n = plan.n, columns = n / 2 + 1;
    const int c = xcd_range(blockIdx.x, columns);
    if (c >= columns) return;
    for (int f = t; f < n; f += kConv) {
        const int r = f - yoff < 0 ? f - yoff + n : f - yoff;
        line[slot(f)] = r < rows ? mid[mid_at(c, r >> 1, pairs) + (r & 1)] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    line_fft<-1, MAXN, kConv>(line, plan, tw, t);
    double2* const k = spectrum + (size_t)c * n;
    if (SPECTRUM) {
        for (int f = t; f < n; f += kConv) {
            const double2 v = line[slot(f)];
            k[f] = make_double2(v.x * scale, v.y * scale);
        }
        return;
    }
    for (int f = t; f < n; f += kConv) line[slot(f)] = cmul(line[slot(f)], k[f]);
    __syncthreads();
    line_fft<1, MAXN, kConv>(line, plan, tw, t);
    // yoff is 0 here; an odd last row's partner is read by nobody
    for (int r = t; r < rows; r += kConv) mid[mid_at(c, r >> 1, pairs) + (r & 1)] = line[slot(r)];
}

// Result rows 2 b and 2 b + 1.
template <int MAXN>
__global__ __launch_bounds__(kConv) void conv_result_kernel(const double2* mid, int rows, int cols, LinePlan plan,
                                                            const double2* tw, int pairs, float* out) {
    __shared__ double2 line[line_slots(MAXN)];
    const int t = threadIdx.x, n = plan.n, h = n / 2;
    const int b = xcd_range(blockIdx.x, pairs);
    if (b >= pairs) return;
    const int y0 = 2 * b;
    const bool two = y0 + 1 < rows;
    for (int f = t; f <= h; f += kConv) {
        const double2* i = mid + mid_at(f, b, pairs);
        const double2 a = i[0], c = two ? i[1] : make_double2(0.0, 0.0);
        line[slot(f)] = make_double2(a.x - c.y, a.y + c.x);
        if (f > 0 && f < h) line[slot(n - f)] = make_double2(a.x + c.y, c.x - a.y);
    }
    __syncthreads();
    line_fft<1, MAXN, kConv>(line, plan, tw, t);
    for (int x = t; x < cols; x += kConv) {
        const double2 v = line[slot(x)];
        out[(size_t)y0 * cols + x] = (float)v.x;
        if (two) out[(size_t)(y0 + 1) * cols + x] = (float)v.y;
    }
}

}  // namespace dev

bool conv_line_plan(int least, LinePlan& p) {
    for (int n = std::max(16, least + least % 2); n <= kMaxLine; n += 2)
        if (line_plan(n, p, true)) return true;
    return false;
}

namespace {
unsigned over_xcds(int n) { return (unsigned)((n + 7) / 8 * 8); }
}  // namespace

hipError_t launch_conv_spectrum(const float* psf, int rows, int cols, int yoff, int xoff, const LinePlan& p,
                                const double2* tw, double2* mid, double2* spectrum, hipStream_t st) {
    const int pairs = (rows + 1) / 2;
    const double scale = 1.0 / ((double)p.n * (double)p.n);
#define P9_ROWS(N)                                                                                                     \
    hipLaunchKernelGGL((dev::conv_rows_kernel<N, true>), dim3(over_xcds(pairs)), dim3(dev::kConv), 0, st, psf, rows, cols, \
                       xoff, p, tw, pairs, mid)
#define P9_COLS(N)                                                                                                            \
    hipLaunchKernelGGL((dev::conv_columns_kernel<N, true>), dim3(over_xcds(p.n / 2 + 1)), dim3(dev::kConv), 0, st, mid, rows, \
                       yoff, p, tw, pairs, scale, spectrum)
    P9_LINE(P9_ROWS);
    if (hipError_t e = hipGetLastError()) return e;
    P9_LINE(P9_COLS);
#undef P9_ROWS
#undef P9_COLS
    return hipGetLastError();
}

hipError_t launch_conv(const float* img, int rows, int cols, const LinePlan& p, const double2* tw, double2* mid,
                       const double2* spectrum, float* out, hipStream_t st) {
    const int pairs = (rows + 1) / 2;
    double2* const k = const_cast<double2*>(spectrum);  // read only
#define P9_ROWS(N)                                                                                                      \
    hipLaunchKernelGGL((dev::conv_rows_kernel<N, false>), dim3(over_xcds(pairs)), dim3(dev::kConv), 0, st, img, rows, cols, \
                       0, p, tw, pairs, mid)
#define P9_COLS(N)                                                                                                             \
    hipLaunchKernelGGL((dev::conv_columns_kernel<N, false>), dim3(over_xcds(p.n / 2 + 1)), dim3(dev::kConv), 0, st, mid, rows, \
                       0, p, tw, pairs, 1.0, k)
#define P9_RESULT(N)                                                                                                   \
    hipLaunchKernelGGL((dev::conv_result_kernel<N>), dim3(over_xcds(pairs)), dim3(dev::kConv), 0, st, mid, rows, cols, \
                       p, tw, pairs, out)
    P9_LINE(P9_ROWS);
    if (hipError_t e = hipGetLastError()) return e;
    P9_LINE(P9_COLS);
    if (hipError_t e = hipGetLastError()) return e;
    P9_LINE(P9_RESULT);
#undef P9_ROWS
#undef P9_COLS
#undef P9_RESULT
    return hipGetLastError();
}

}  // namespace p9idg
