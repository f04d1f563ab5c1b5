// The grid <-> image transforms between the w-stack and the image
// (FFT.cs:99-117, :188-215, :248-264) for even G = 2^a 3^b 5^c up to 4096, on
// Stockham FFTs in LDS.  The image side is real and, towards the image, the
// grid is zero outside the subgrids' bounding box, so
//   ToImage  transforms only the box's columns (v -> y), then pairs of rows
//            (u -> x) whose Hermitian parts share one complex transform:
//            Re(IFFT) of two rows at once, written as whole image rows;
//   ToUVW    transforms pairs of real image rows with one complex transform,
//            keeps the G / 2 + 1 columns that determine the rest, transforms
//            them and writes each with its conjugate mirror.
// A 2-D library transform moves the complex grid four times (read + write per
// pass, 75 MB each way at 3072^2) besides the real <-> complex copies.
#include "p9idg_internal.h"

namespace p9idg {
namespace dev {

constexpr int kLine = 256;  // threads of one line

// LDS index of element i: a gap every 16 elements spreads the radix strides
// over the banks.
__device__ __forceinline__ int slot(int i) { return i + (i >> 4); }
constexpr int line_slots(int n) { return n + n / 16 + 1; }

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) { return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
// sign * i * a
template <int SIGN>
__device__ __forceinline__ float2 ci(float2 a) {
    return SIGN > 0 ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

// R-point transforms with kernel exp(SIGN 2 pi i / R), in natural order.
template <int SIGN>
__device__ __forceinline__ void dft2(float2& a, float2& b) {
    const float2 t = a;
    a = cadd(t, b);
    b = csub(t, b);
}
template <int SIGN>
__device__ __forceinline__ void dft4(float2& a, float2& b, float2& c, float2& d) {
    const float2 s02 = cadd(a, c), d02 = csub(a, c), s13 = cadd(b, d), d13 = ci<SIGN>(csub(b, d));
    a = cadd(s02, s13);
    b = cadd(d02, d13);
    c = csub(s02, s13);
    d = csub(d02, d13);
}
template <int R, int SIGN>
struct Dft;
template <int SIGN>
struct Dft<2, SIGN> {
    __device__ static __forceinline__ void run(float2* v) { dft2<SIGN>(v[0], v[1]); }
};
template <int SIGN>
struct Dft<4, SIGN> {
    __device__ static __forceinline__ void run(float2* v) { dft4<SIGN>(v[0], v[1], v[2], v[3]); }
};
template <int SIGN>
struct Dft<3, SIGN> {
    __device__ static __forceinline__ void run(float2* v) {
        constexpr float h = 0.86602540378443864676f;  // sqrt(3) / 2
        const float2 t = cadd(v[1], v[2]), d = ci<SIGN>(csub(v[1], v[2]));
        const float2 m = make_float2(v[0].x - 0.5f * t.x, v[0].y - 0.5f * t.y);
        v[0] = cadd(v[0], t);
        v[1] = make_float2(m.x + h * d.x, m.y + h * d.y);
        v[2] = make_float2(m.x - h * d.x, m.y - h * d.y);
    }
};
template <int SIGN>
struct Dft<5, SIGN> {
    __device__ static __forceinline__ void run(float2* v) {
        // cos and sin of 2 pi / 5 and 4 pi / 5
        constexpr float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
        constexpr float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;
        const float2 a = cadd(v[1], v[4]), b = cadd(v[2], v[3]);
        const float2 p = ci<SIGN>(csub(v[1], v[4])), q = ci<SIGN>(csub(v[2], v[3]));
        const float2 m1 = make_float2(v[0].x + c1 * a.x + c2 * b.x, v[0].y + c1 * a.y + c2 * b.y);
        const float2 m2 = make_float2(v[0].x + c2 * a.x + c1 * b.x, v[0].y + c2 * a.y + c1 * b.y);
        const float2 n1 = make_float2(s1 * p.x + s2 * q.x, s1 * p.y + s2 * q.y);
        const float2 n2 = make_float2(s2 * p.x - s1 * q.x, s2 * p.y - s1 * q.y);
        v[0] = cadd(v[0], cadd(a, b));
        v[1] = cadd(m1, n1);
        v[4] = csub(m1, n1);
        v[2] = cadd(m2, n2);
        v[3] = csub(m2, n2);
    }
};
// 16 = 4 x 4: columns, the inner twiddles exp(SIGN 2 pi i r c / 16), rows
template <int SIGN>
struct Dft<16, SIGN> {
    __device__ static __forceinline__ void run(float2* v) {
        constexpr float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f, c2 = 0.70710678118654752440f;
        auto w = [](float c, float s) { return make_float2(c, SIGN > 0 ? s : -s); };
#pragma unroll
        for (int r = 0; r < 4; r++) dft4<SIGN>(v[r], v[r + 4], v[r + 8], v[r + 12]);
        v[5] = cmul(v[5], w(c1, s1));
        v[6] = cmul(v[6], w(c2, c2));
        v[7] = cmul(v[7], w(s1, c1));
        v[9] = cmul(v[9], w(c2, c2));
        v[10] = ci<SIGN>(v[10]);
        v[11] = cmul(v[11], w(-c2, c2));
        v[13] = cmul(v[13], w(s1, c1));
        v[14] = cmul(v[14], w(-c2, c2));
        v[15] = cmul(v[15], w(-c1, -s1));
        float2 o[16];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            dft4<SIGN>(v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]);
#pragma unroll
            for (int q = 0; q < 4; q++) o[r + 4 * q] = v[4 * r + q];
        }
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = o[i];
    }
};
template <int SIGN>
struct Dft<8, SIGN> {
    __device__ static __forceinline__ void run(float2* v) {
        constexpr float c2 = 0.70710678118654752440f;
        auto w = [](float c, float s) { return make_float2(c, SIGN > 0 ? s : -s); };
        dft4<SIGN>(v[0], v[2], v[4], v[6]);
        dft4<SIGN>(v[1], v[3], v[5], v[7]);
        const float2 t1 = cmul(v[3], w(c2, c2)), t2 = ci<SIGN>(v[5]), t3 = cmul(v[7], w(-c2, c2));
        const float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1];
        v[0] = cadd(e0, o0);
        v[4] = csub(e0, o0);
        v[1] = cadd(e1, t1);
        v[5] = csub(e1, t1);
        v[2] = cadd(e2, t2);
        v[6] = csub(e2, t2);
        v[3] = cadd(e3, t3);
        v[7] = csub(e3, t3);
    }
};

// One Stockham pass of radix R over a line of n elements by kLine threads, in
// place: every butterfly is read before any is written.  tw[k] = exp(2 pi i k / n).
template <int R, int SIGN, int MAXN>
__device__ __forceinline__ void line_pass(float2* line, int n, int Ns, const float2* tw, int t) {
    constexpr int IT = (MAXN / R + kLine - 1) / kLine;
    const int M = n / R, stride = n / (Ns * R);
    float2 v[IT][R];
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int j = t + i * kLine;
        if (j < M)
#pragma unroll
            for (int q = 0; q < R; q++) v[i][q] = line[slot(j + q * M)];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int j = t + i * kLine;
        if (j < M) {
            const int d = j / Ns, k = j - d * Ns;
            if (Ns > 1)
#pragma unroll
                for (int q = 1; q < R; q++) {
                    float2 w = tw[q * k * stride];  // < n
                    if (SIGN < 0) w.y = -w.y;
                    v[i][q] = cmul(v[i][q], w);
                }
            Dft<R, SIGN>::run(v[i]);
            const int base = d * Ns * R + k;
#pragma unroll
            for (int q = 0; q < R; q++) line[slot(base + q * Ns)] = v[i][q];
        }
    }
    __syncthreads();
}
// The whole line; its elements are in place and every thread has passed a barrier.
template <int SIGN, int MAXN>
__device__ __forceinline__ void line_fft(float2* line, const LinePlan& p, const float2* tw, int t) {
    int Ns = 1;
    for (int i = 0; i < p.passes; i++) {  // uniform
        const int R = p.radix[i];
        switch (R) {
            case 16: line_pass<16, SIGN, MAXN>(line, p.n, Ns, tw, t); break;
            case 8: line_pass<8, SIGN, MAXN>(line, p.n, Ns, tw, t); break;
            case 4: line_pass<4, SIGN, MAXN>(line, p.n, Ns, tw, t); break;
            case 2: line_pass<2, SIGN, MAXN>(line, p.n, Ns, tw, t); break;
            case 5: line_pass<5, SIGN, MAXN>(line, p.n, Ns, tw, t); break;
            default: line_pass<3, SIGN, MAXN>(line, p.n, Ns, tw, t); break;
        }
        Ns *= R;
    }
}

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

// ToImage, columns: column u.x0 + c of the box (dense array, or the
// quadrant-swapped grid) over v; mid[y][c] for every storage row y.
template <int MAXN, int LINES>
__global__ __launch_bounds__(kLine * LINES) void image_columns_kernel(const float2* src, bool dense, Box u, LinePlan plan,
                                                                      const float2* tw, float2* mid) {
    __shared__ float2 s_line[LINES][line_slots(MAXN)];
    const int t = threadIdx.x % kLine, l = threadIdx.x / kLine, G = plan.n, h = G / 2;
    const int w = u.x1 - u.x0, c = blockIdx.x * LINES + l;
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
    line_fft<1, MAXN>(line, plan, tw, t);
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
__global__ __launch_bounds__(kLine) void image_rows_kernel(const float2* mid, Box u, LinePlan plan, const float2* tw,
                                                           double inv_n, float* img) {
    __shared__ float2 line[line_slots(MAXN)];
    const int t = threadIdx.x, G = plan.n, h = G / 2, w = u.x1 - u.x0;
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
    line_fft<1, MAXN>(line, plan, tw, t);
    float* o0 = img + (size_t)(y0 >= h ? y0 - h : y0 + h) * G;
    float* o1 = img + (size_t)(y1 >= h ? y1 - h : y1 + h) * G;
    for (int x = t; x < G; x += kLine) {
        const float2 v = line[slot(x)];
        const int at = x >= h ? x - h : x + h;
        o0[at] = (float)((double)v.x * inv_n);
        o1[at] = (float)((double)v.y * inv_n);
    }
}

// ToUVW, rows: storage rows 2 b and 2 b + 1 of the quadrant-swapped image;
// mid[y][f] for f = 0 .. G / 2 (row pitch `pitch`).
template <int MAXN>
__global__ __launch_bounds__(kLine) void grid_rows_kernel(const float* img, LinePlan plan, const float2* tw, int pitch,
                                                          float2* mid) {
    __shared__ float2 line[line_slots(MAXN)];
    const int t = threadIdx.x, G = plan.n, h = G / 2;
    const int y0 = 2 * blockIdx.x, y1 = y0 + 1;
    const float* i0 = img + (size_t)(y0 >= h ? y0 - h : y0 + h) * G;
    const float* i1 = img + (size_t)(y1 >= h ? y1 - h : y1 + h) * G;
    for (int x = t; x < G; x += kLine) {
        const int at = x >= h ? x - h : x + h;
        line[slot(x)] = make_float2(i0[at], i1[at]);
    }
    __syncthreads();
    line_fft<-1, MAXN>(line, plan, tw, t);
    for (int f = t; f <= h; f += kLine) {
        const float2 z = line[slot(f)], c = line[slot(f ? G - f : 0)];
        mid[(size_t)y0 * pitch + f] = make_float2(0.5f * (z.x + c.x), 0.5f * (z.y - c.y));
        mid[(size_t)y1 * pitch + f] = make_float2(0.5f * (z.y + c.y), 0.5f * (c.x - z.x));
    }
}
// ToUVW, columns: columns f and their mirrors G - f.
template <int MAXN, int LINES>
__global__ __launch_bounds__(kLine * LINES) void grid_columns_kernel(const float2* mid, int pitch, LinePlan plan,
                                                                     const float2* tw, float2* grid) {
    __shared__ float2 s_line[LINES][line_slots(MAXN)];
    const int G = plan.n, h = G / 2;
    // workgroups go round robin over the 8 XCDs: give each XCD neighbouring
    // columns, whose lines its L2 then holds for all of them
    const int per = (gridDim.x + 7) / 8, blk = (blockIdx.x % 8) * per + blockIdx.x / 8;
    const int f0 = blk * LINES, cols = min(LINES, h + 1 - f0);
    if (cols <= 0) return;  // whole workgroups
    for (int i = threadIdx.x; i < G * LINES; i += kLine * LINES) {
        const int y = i / LINES, k = i % LINES;
        s_line[k][slot(y)] = k < cols ? mid[(size_t)y * pitch + f0 + k] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    line_fft<-1, MAXN>(s_line[threadIdx.x / kLine], plan, tw, threadIdx.x % kLine);
    for (int i = threadIdx.x; i < G * LINES; i += kLine * LINES) {
        const int v = i / LINES, k = i % LINES, f = f0 + k;
        if (k >= cols) continue;
        const float2 e = s_line[k][slot(v)];
        grid[(size_t)v * G + f] = e;
        if (f > 0 && f < h) grid[(size_t)(v ? G - v : 0) * G + G - f] = make_float2(e.x, -e.y);
    }
}

}  // namespace dev

bool line_plan(int n, LinePlan& p) {
    p = LinePlan{};
    if (n < 16 || n > kMaxLine || n % 2) return false;
    p.n = n;
    for (int r : {16, 8, 4, 2, 5, 3})
        while (n % r == 0 && p.passes < kMaxPasses) {
            p.radix[p.passes++] = r;
            n /= r;
        }
    return n == 1;
}

// LDS is sized for the next power of two.
#define P9_LINE(CALL)              \
    do {                           \
        if (p.n <= 512) {          \
            CALL(512);             \
        } else if (p.n <= 1024) {  \
            CALL(1024);            \
        } else if (p.n <= 2048) {  \
            CALL(2048);            \
        } else if (p.n <= 3072) {  \
            CALL(3072);            \
        } else {                   \
            CALL(4096);            \
        }                          \
    } while (0)

hipError_t launch_sum_boxes(const float2* layers, const Box* boxes, int nboxes, int G, Box u, float2* out, hipStream_t st) {
    const int n = (u.y1 - u.y0) * (u.x1 - u.x0);
    hipLaunchKernelGGL(dev::sum_boxes_kernel, dim3((n + 255) / 256), dim3(256), 0, st, layers, boxes, nboxes, G, u, out);
    return hipGetLastError();
}

hipError_t launch_line_image(const float2* src, bool dense, Box u, const LinePlan& p, const float2* tw, float2* mid,
                             double inv_n, float* img, hipStream_t st) {
    constexpr int L = 2;
    const int w = u.x1 - u.x0;
#define P9_COLS(N)                                                                                                      \
    hipLaunchKernelGGL((dev::image_columns_kernel<N, L>), dim3((w + L - 1) / L), dim3(dev::kLine * L), 0, st, src, dense, u, \
                       p, tw, mid)
#define P9_ROWS(N) \
    hipLaunchKernelGGL((dev::image_rows_kernel<N>), dim3(p.n / 2), dim3(dev::kLine), 0, st, mid, u, p, tw, inv_n, img)
    P9_LINE(P9_COLS);
    if (hipError_t e = hipGetLastError()) return e;
    P9_LINE(P9_ROWS);
#undef P9_COLS
#undef P9_ROWS
    return hipGetLastError();
}

hipError_t launch_line_grid(const float* img, const LinePlan& p, const float2* tw, float2* mid, float2* grid, hipStream_t st) {
    constexpr int L = 4;
    const int pitch = line_pitch(p.n);
#define P9_ROWS(N) \
    hipLaunchKernelGGL((dev::grid_rows_kernel<N>), dim3(p.n / 2), dim3(dev::kLine), 0, st, img, p, tw, pitch, mid)
#define P9_COLS(N)                                                                                                           \
    hipLaunchKernelGGL((dev::grid_columns_kernel<N, L>), dim3(((p.n / 2 + 1 + L - 1) / L + 7) / 8 * 8), dim3(dev::kLine * L), 0, \
                       st, mid, pitch, p, tw, grid)
    P9_LINE(P9_ROWS);
    if (hipError_t e = hipGetLastError()) return e;
    P9_LINE(P9_COLS);
#undef P9_COLS
#undef P9_ROWS
    return hipGetLastError();
}

}  // namespace p9idg
