// The grid <-> image transforms between the w-stack and the image
// (FFT.cs:99-117, :188-215, :248-264) for even G = 2^a 3^b 5^c up to 4096, on
// Stockham FFTs in LDS.  The image side is real and, towards the image, the
// grid is zero outside the subgrids' bounding box, so
//   ToImage  transforms only the box's columns (v -> y), then pairs of rows
//            (u -> x) whose Hermitian parts share one complex transform:
//            Re(IFFT) of two rows at once, written as whole image rows;
//   ToUVW    transforms pairs of real image columns with one complex transform,
//            keeps the G / 2 + 1 rows that determine the rest, transforms them
//            and writes each with its conjugate mirror.
// A 2-D library transform moves the complex grid four times (read + write per
// pass, 75 MB each way at 3072^2) besides the real <-> complex copies.
#include "device_linefft.h"

namespace p9idg {
namespace dev {

constexpr int kLine = 256;  // threads of one line

// Sum of the w-layers over the union box u of their footprints, as a dense
// (u.y1 - u.y0) x (u.x1 - u.x0) array.
__global__ void sum_boxes_kernel(const float2* layers, const Box* boxes, int nboxes, int G, Box u, float2* out) {
    const int w = u.x1 - u.x0, n = (u.y1 - u.y0) * w, h = G / 2;
    const size_t GG = (size_t)G * G;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int y = u.y0 + i / w, x = u.x0 + i % w;
        const size_t idx = (size_t)(y >= h ? y - h : y + h) * G + (x >= h ? x - h : x + h);
        float2 acc = make_float2(0.f, 0.f);
        for (int b = 0; b < nboxes; b++) {
            const Box bx = boxes[b];
            if (y >= bx.y0 && y < bx.y1 && x >= bx.x0 && x < bx.x1) acc = cadd(acc, layers[bx.layer * GG + idx]);
        }
        out[i] = acc;
    }
}

// *wide: whether the quadrant-swapped grid holds anything outside u (storage
// row blockIdx.x); *next, the following check's word, is cleared.  The grid of a
// caller that writes into it from time to time is read once (75 MB at 3072^2)
// instead of transformed over its whole width: gridding and image 2048^2 132 -> 83
// us, 3072^2 243 -> 102 (the box alone, unchecked: 61 and 77).
__global__ __launch_bounds__(kLine) void outside_kernel(const float2* grid, int G, Box u, int32_t* wide, int32_t* next) {
    const int h = G / 2, f = blockIdx.x, v = f >= h ? f - h : f + h;
    const bool row = v >= u.y0 && v < u.y1;
    const float4* in = reinterpret_cast<const float4*>(grid + (size_t)f * G);  // G is even
    bool any = false;
    for (int i = threadIdx.x; i < h; i += kLine) {
        const uint4 e = __builtin_bit_cast(uint4, in[i]);
        const int c = 2 * i, x0 = c >= h ? c - h : c + h, x1 = c + 1 >= h ? c + 1 - h : c + 1 + h;
        any |= !(row && x0 >= u.x0 && x0 < u.x1) && (e.x | e.y);
        any |= !(row && x1 >= u.x0 && x1 < u.x1) && (e.z | e.w);
    }
    if (__syncthreads_or(any) && threadIdx.x == 0) *wide = 1;
    if (f == 0 && threadIdx.x == 0) *next = 0;
}
__device__ __forceinline__ Box box_of(Box u, const int32_t* wide, int G) { return wide && *wide ? Box{0, 0, G, 0, G} : u; }

// ToImage, columns: column u.x0 + c of the box (dense array, or the
// quadrant-swapped grid) over v; mid[y][c] for every storage row y.  wide: the
// box is the whole grid where that word is set.
template <int MAXN, int LINES>
__global__ __launch_bounds__(kLine * LINES) void image_columns_kernel(const float2* src, bool dense, Box box, const int32_t* wide,
                                                                                   LinePlan plan, const float2* tw,
                                                                                   float2* mid) {
    __shared__ float2 s_line[LINES][line_slots(MAXN)];
    const int t = threadIdx.x % kLine, l = threadIdx.x / kLine, G = plan.n, h = G / 2;
    const Box u = box_of(box, wide, G);
    const int w = u.x1 - u.x0, c = blockIdx.x * LINES + l;
    if ((int)blockIdx.x * LINES >= w) return;  // whole workgroups
    float2* line = s_line[l];
    for (int f = t; f < G; f += kLine) {
        const int v = f >= h ? f - h : f + h;  // grid row of frequency f
        float2 e = make_float2(0.f, 0.f);
        if (c < w && v >= u.y0 && v < u.y1) {
            const int x = u.x0 + c;
            e = dense ? src[(v - u.y0) * w + c] : src[(size_t)f * G + (x >= h ? x - h : x + h)];
        }
        line[slot(f)] = e;
    }
    __syncthreads();
    line_fft<1, MAXN, kLine>(line, plan, tw, t);
    // neighbouring threads write a row's neighbouring columns
    const int cols = min(LINES, w - (int)blockIdx.x * LINES);
    for (int i = threadIdx.x; i < G * LINES; i += kLine * LINES) {
        const int y = i / LINES, k = i % LINES;
        if (k < cols) mid[(size_t)y * w + blockIdx.x * LINES + k] = s_line[k][slot(y)];
    }
}
// ToImage, rows: storage rows 2 b and 2 b + 1 over u; image rows scaled by
// inv_n, quadrant-swapped.
template <int MAXN>
__global__ __launch_bounds__(kLine) void image_rows_kernel(const float2* mid, Box box, const int32_t* wide, LinePlan plan,
                                                                        const float2* tw, double inv_n, float* img) {
    __shared__ float2 line[line_slots(MAXN)];
    const int t = threadIdx.x, G = plan.n, h = G / 2;
    const Box u = box_of(box, wide, G);
    const int w = u.x1 - u.x0;
    const int y0 = 2 * blockIdx.x, y1 = y0 + 1;  // G is even
    const float2* r0 = mid + (size_t)y0 * w;
    const float2* r1 = r0 + w;
    for (int f = t; f < G; f += kLine) {
        // Hermitian part (A[f] + conj A[-f]) / 2 of both rows, as a + i b
        const int g = f ? G - f : 0;
        const int xf = (f >= h ? f - h : f + h) - u.x0, xg = (g >= h ? g - h : g + h) - u.x0;
        float2 z = make_float2(0.f, 0.f);
        if (xf >= 0 && xf < w) {
            const float2 a = r0[xf], b = r1[xf];
            z = make_float2(a.x - b.y, a.y + b.x);
        }
        if (xg >= 0 && xg < w) {
            const float2 a = r0[xg], b = r1[xg];
            z = make_float2(z.x + a.x + b.y, z.y - a.y + b.x);
        }
        line[slot(f)] = make_float2(0.5f * z.x, 0.5f * z.y);
    }
    __syncthreads();
    line_fft<1, MAXN, kLine>(line, plan, tw, t);
    float* o0 = img + (size_t)(y0 >= h ? y0 - h : y0 + h) * G;
    float* o1 = img + (size_t)(y1 >= h ? y1 - h : y1 + h) * G;
    for (int x = t; x < G; x += kLine) {
        const float2 v = line[slot(x)];
        const int at = x >= h ? x - h : x + h;
        o0[at] = (float)((double)v.x * inv_n);
        o1[at] = (float)((double)v.y * inv_n);
    }
}

// ToUVW, columns: LINES pairs of real columns of the quadrant-swapped image, a
// pair as one complex line; mid[f][x] for f = 0 .. G / 2.  The grid's rows are
// then written whole: with the rows first, the columns' 32-byte pieces of the
// grid and of its mirror were the larger half of the time (4096^2 182 -> 133
// us, 3072^2 87 -> 76, 2048^2 59 -> 45).
template <int MAXN, int LINES>
__global__ __launch_bounds__(kLine * LINES) void grid_columns_kernel(const float* img, LinePlan plan,
                                                                                  const float2* tw, float2* mid) {
    __shared__ float2 s_line[LINES][line_slots(MAXN)];
    const int G = plan.n, h = G / 2;
    // workgroups go round robin over the 8 XCDs: give each XCD neighbouring
    // columns, whose lines its L2 then holds for all of them
    const int per = (gridDim.x + 7) / 8, blk = (blockIdx.x % 8) * per + blockIdx.x / 8;
    const int c0 = blk * LINES, lines = min(LINES, h - c0);  // column pairs
    if (lines <= 0) return;  // whole workgroups
    for (int i = threadIdx.x; i < G * LINES; i += kLine * LINES) {
        const int y = i / LINES, k = i % LINES, x = 2 * (c0 + k);
        float2 e = make_float2(0.f, 0.f);
        if (k < lines) {
            const float* row = img + (size_t)(y >= h ? y - h : y + h) * G;
            e.x = row[x >= h ? x - h : x + h];
            e.y = row[x + 1 >= h ? x + 1 - h : x + 1 + h];
        }
        s_line[k][slot(y)] = e;
    }
    __syncthreads();
    line_fft<-1, MAXN, kLine>(s_line[threadIdx.x / kLine], plan, tw, threadIdx.x % kLine);
    for (int i = threadIdx.x; i < (h + 1) * LINES; i += kLine * LINES) {
        const int f = i / LINES, k = i % LINES;
        if (k >= lines) continue;
        const float2 z = s_line[k][slot(f)], c = s_line[k][slot(f ? G - f : 0)];
        float2* o = mid + (size_t)f * G + 2 * (c0 + k);
        o[0] = make_float2(0.5f * (z.x + c.x), 0.5f * (z.y - c.y));
        o[1] = make_float2(0.5f * (z.y + c.y), 0.5f * (c.x - z.x));
    }
}
// ToUVW, rows: grid row f and its conjugate mirror G - f.
template <int MAXN>
__global__ __launch_bounds__(kLine) void grid_rows_kernel(const float2* mid, LinePlan plan, const float2* tw,
                                                                       float2* grid) {
    __shared__ float2 line[line_slots(MAXN)];
    const int t = threadIdx.x, G = plan.n, h = G / 2, f = blockIdx.x;
    const float2* in = mid + (size_t)f * G;
    for (int x = t; x < G; x += kLine) line[slot(x)] = in[x];
    __syncthreads();
    line_fft<-1, MAXN, kLine>(line, plan, tw, t);
    float2* o = grid + (size_t)f * G;
    for (int u = t; u < G; u += kLine) o[u] = line[slot(u)];
    if (f == 0 || f == h) return;
    float2* m = grid + (size_t)(G - f) * G;
    for (int u = t; u < G; u += kLine) {
        const float2 e = line[slot(u ? G - u : 0)];
        m[u] = make_float2(e.x, -e.y);
    }
}

}  // namespace dev

bool line_plan(int n, LinePlan& p, bool nine) {
    p = LinePlan{};
    if (n < 16 || n > kMaxLine || n % 2) return false;
    p.n = n;
    for (int r : {16, 9, 8, 4, 2, 5, 3})
        while (n % r == 0 && p.passes < kMaxPasses && (r != 9 || nine)) {
            p.radix[p.passes++] = r;
            n /= r;
        }
    return n == 1;
}

hipError_t launch_sum_boxes(const float2* layers, const Box* boxes, int nboxes, int G, Box u, float2* out, hipStream_t st) {
    const int n = (u.y1 - u.y0) * (u.x1 - u.x0);
    hipLaunchKernelGGL(dev::sum_boxes_kernel, dim3((n + 255) / 256), dim3(256), 0, st, layers, boxes, nboxes, G, u, out);
    return hipGetLastError();
}

hipError_t launch_outside(const float2* grid, Box u, int G, int32_t* wide, int32_t* next, hipStream_t st) {
    hipLaunchKernelGGL(dev::outside_kernel, dim3(G), dim3(dev::kLine), 0, st, grid, G, u, wide, next);
    return hipGetLastError();
}

hipError_t launch_line_image(const float2* src, bool dense, Box u, const int32_t* wide, const LinePlan& p, const float2* tw,
                             float2* mid, double inv_n, float* img, hipStream_t st) {
    constexpr int L = 2;
    const int w = wide ? p.n : u.x1 - u.x0;
#define P9_COLS(N)                                                                                                      \
    hipLaunchKernelGGL((dev::image_columns_kernel<N, L>), dim3((w + L - 1) / L), dim3(dev::kLine * L), 0, st, src, dense, u, \
                       wide, p, tw, mid)
#define P9_ROWS(N) \
    hipLaunchKernelGGL((dev::image_rows_kernel<N>), dim3(p.n / 2), dim3(dev::kLine), 0, st, mid, u, wide, p, tw, inv_n, img)
    P9_LINE(P9_COLS);
    if (hipError_t e = hipGetLastError()) return e;
    P9_LINE(P9_ROWS);
#undef P9_COLS
#undef P9_ROWS
    return hipGetLastError();
}

hipError_t launch_line_grid(const float* img, const LinePlan& p, const float2* tw, float2* mid, float2* grid, hipStream_t st) {
    constexpr int L = 2;  // 3072^2: as many workgroups as the chip holds; 4: 88 us
    const unsigned blocks = ((p.n / 2 + L - 1) / L + 7) / 8 * 8;
#define P9_COLS(N) \
    hipLaunchKernelGGL((dev::grid_columns_kernel<N, L>), dim3(blocks), dim3(dev::kLine * L), 0, st, img, p, tw, mid)
#define P9_ROWS(N) hipLaunchKernelGGL((dev::grid_rows_kernel<N>), dim3(p.n / 2 + 1), dim3(dev::kLine), 0, st, mid, p, tw, grid)
    P9_LINE(P9_COLS);
    if (hipError_t e = hipGetLastError()) return e;
    P9_LINE(P9_ROWS);
#undef P9_COLS
#undef P9_ROWS
    return hipGetLastError();
}

}  // namespace p9idg
