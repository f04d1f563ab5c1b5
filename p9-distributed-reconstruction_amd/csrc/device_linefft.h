// Stockham FFTs of one line in LDS, FP32 (float2) or FP64 (double2), for
// lengths n = 2^a 3^b 5^c up to 4096 (kernels_fft.hip, kernels_conv.hip).
#pragma once

#include "p9idg_internal.h"

namespace p9idg {
namespace dev {

// LDS index of element i: a gap every 16 elements spreads the radix strides
// over the banks.
__device__ __forceinline__ int slot(int i) { return i + (i >> 4); }
constexpr int line_slots(int n) { return n + n / 16 + 1; }

template <typename V>
struct Real;
template <>
struct Real<float2> {
    using T = float;
};
template <>
struct Real<double2> {
    using T = double;
};
template <typename V>
__device__ __forceinline__ V make(typename Real<V>::T x, typename Real<V>::T y) {
    V v;
    v.x = x;
    v.y = y;
    return v;
}
template <typename V>
__device__ __forceinline__ V cadd(V a, V b) {
    return make<V>(a.x + b.x, a.y + b.y);
}
template <typename V>
__device__ __forceinline__ V csub(V a, V b) {
    return make<V>(a.x - b.x, a.y - b.y);
}
template <typename V>
__device__ __forceinline__ V cmul(V a, V b) {
    return make<V>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// sign * i * a
template <int SIGN, typename V>
__device__ __forceinline__ V ci(V a) {
    return SIGN > 0 ? make<V>(-a.y, a.x) : make<V>(a.y, -a.x);
}

// R-point transforms with kernel exp(SIGN 2 pi i / R), in natural order.
template <typename V>
__device__ __forceinline__ void dft2(V& a, V& b) {
    const V t = a;
    a = cadd(t, b);
    b = csub(t, b);
}
template <int SIGN, typename V>
__device__ __forceinline__ void dft3(V& a, V& b, V& c) {
    using T = typename Real<V>::T;
    constexpr T h = (T)0.86602540378443864676;  // sqrt(3) / 2
    const V t = cadd(b, c), d = ci<SIGN>(csub(b, c));
    const V m = make<V>(a.x - (T)0.5 * t.x, a.y - (T)0.5 * t.y);
    a = cadd(a, t);
    b = make<V>(m.x + h * d.x, m.y + h * d.y);
    c = make<V>(m.x - h * d.x, m.y - h * d.y);
}
template <int SIGN, typename V>
__device__ __forceinline__ void dft4(V& a, V& b, V& c, V& d) {
    const V s02 = cadd(a, c), d02 = csub(a, c), s13 = cadd(b, d), d13 = ci<SIGN>(csub(b, d));
    a = cadd(s02, s13);
    b = cadd(d02, d13);
    c = csub(s02, s13);
    d = csub(d02, d13);
}
template <int R, int SIGN, typename V>
__device__ __forceinline__ void dft(V* v) {
    using T = typename Real<V>::T;
    auto w = [](T c, T s) { return make<V>(c, SIGN > 0 ? s : -s); };
    if constexpr (R == 2) {
        dft2(v[0], v[1]);
    } else if constexpr (R == 3) {
        dft3<SIGN>(v[0], v[1], v[2]);
    } else if constexpr (R == 4) {
        dft4<SIGN>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 5) {
        // cos and sin of 2 pi / 5 and 4 pi / 5
        constexpr T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
        constexpr T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;
        const V a = cadd(v[1], v[4]), b = cadd(v[2], v[3]);
        const V p = ci<SIGN>(csub(v[1], v[4])), q = ci<SIGN>(csub(v[2], v[3]));
        const V m1 = make<V>(v[0].x + c1 * a.x + c2 * b.x, v[0].y + c1 * a.y + c2 * b.y);
        const V m2 = make<V>(v[0].x + c2 * a.x + c1 * b.x, v[0].y + c2 * a.y + c1 * b.y);
        const V n1 = make<V>(s1 * p.x + s2 * q.x, s1 * p.y + s2 * q.y);
        const V n2 = make<V>(s2 * p.x - s1 * q.x, s2 * p.y - s1 * q.y);
        v[0] = cadd(v[0], cadd(a, b));
        v[1] = cadd(m1, n1);
        v[4] = csub(m1, n1);
        v[2] = cadd(m2, n2);
        v[3] = csub(m2, n2);
    } else if constexpr (R == 8) {
        constexpr T c2 = (T)0.70710678118654752440;
        dft4<SIGN>(v[0], v[2], v[4], v[6]);
        dft4<SIGN>(v[1], v[3], v[5], v[7]);
        const V t1 = cmul(v[3], w(c2, c2)), t2 = ci<SIGN>(v[5]), t3 = cmul(v[7], w(-c2, c2));
        const V e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1];
        v[0] = cadd(e0, o0);
        v[4] = csub(e0, o0);
        v[1] = cadd(e1, t1);
        v[5] = csub(e1, t1);
        v[2] = cadd(e2, t2);
        v[6] = csub(e2, t2);
        v[3] = cadd(e3, t3);
        v[7] = csub(e3, t3);
    } else if constexpr (R == 9) {
        // 9 = 3 x 3: columns, the inner twiddles exp(SIGN 2 pi i r c / 9), rows
        constexpr T c1 = (T)0.76604444311897803520, s1 = (T)0.64278760968653932632;
        constexpr T c2 = (T)0.17364817766693034885, s2 = (T)0.98480775301220805937;
        constexpr T c4 = (T)-0.93969262078590838405, s4 = (T)0.34202014332566873304;
#pragma unroll
        for (int r = 0; r < 3; r++) dft3<SIGN>(v[r], v[r + 3], v[r + 6]);
        v[4] = cmul(v[4], w(c1, s1));
        v[5] = cmul(v[5], w(c2, s2));
        v[7] = cmul(v[7], w(c2, s2));
        v[8] = cmul(v[8], w(c4, s4));
        V o[9];
#pragma unroll
        for (int r = 0; r < 3; r++) {
            dft3<SIGN>(v[3 * r], v[3 * r + 1], v[3 * r + 2]);
#pragma unroll
            for (int q = 0; q < 3; q++) o[r + 3 * q] = v[3 * r + q];
        }
#pragma unroll
        for (int i = 0; i < 9; i++) v[i] = o[i];
    } else {
        static_assert(R == 16, "radix");
        // 16 = 4 x 4: columns, the inner twiddles exp(SIGN 2 pi i r c / 16), rows
        constexpr T c1 = (T)0.92387953251128675613, s1 = (T)0.38268343236508977173, c2 = (T)0.70710678118654752440;
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
        V o[16];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            dft4<SIGN>(v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]);
#pragma unroll
            for (int q = 0; q < 4; q++) o[r + 4 * q] = v[4 * r + q];
        }
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = o[i];
    }
}

// One Stockham pass of radix R over a line of n elements by NT threads, in
// place: every butterfly is read before any is written.  tw[k] = exp(2 pi i k / n).
// FP32 reads every twiddle from the table; FP64, whose table is as large as the
// line, reads one per butterfly and multiplies up its powers (1e-15).
template <int R, int SIGN, int MAXN, int NT, typename V>
__device__ __forceinline__ void line_pass(V* line, int n, int Ns, const V* tw, int t) {
    constexpr int IT = (MAXN / R + NT - 1) / NT;
    const int M = n / R, stride = n / (Ns * R);
    V v[IT][R];
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int j = t + i * NT;
        if (j < M)
#pragma unroll
            for (int q = 0; q < R; q++) v[i][q] = line[slot(j + q * M)];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int j = t + i * NT;
        if (j < M) {
            const int d = j / Ns, k = j - d * Ns;
            if (Ns > 1) {
                if constexpr (sizeof(V) == sizeof(double2)) {
                    V w1 = tw[k * stride];  // < n / R
                    if (SIGN < 0) w1.y = -w1.y;
                    V w = w1;
#pragma unroll
                    for (int q = 1; q < R; q++) {
                        v[i][q] = cmul(v[i][q], w);
                        if (q + 1 < R) w = cmul(w, w1);
                    }
                } else {
#pragma unroll
                    for (int q = 1; q < R; q++) {
                        V w = tw[q * k * stride];  // < n
                        if (SIGN < 0) w.y = -w.y;
                        v[i][q] = cmul(v[i][q], w);
                    }
                }
            }
            dft<R, SIGN>(v[i]);
            const int base = d * Ns * R + k;
#pragma unroll
            for (int q = 0; q < R; q++) line[slot(base + q * Ns)] = v[i][q];
        }
    }
    __syncthreads();
}
// The whole line; its elements are in place and every thread has passed a barrier.
template <int SIGN, int MAXN, int NT, typename V>
__device__ __forceinline__ void line_fft(V* line, const LinePlan& p, const V* tw, int t) {
    int Ns = 1;
    for (int i = 0; i < p.passes; i++) {  // uniform
        const int R = p.radix[i];
        switch (R) {
            case 16: line_pass<16, SIGN, MAXN, NT>(line, p.n, Ns, tw, t); break;
            case 9:
                if constexpr (sizeof(V) == sizeof(double2)) line_pass<9, SIGN, MAXN, NT>(line, p.n, Ns, tw, t);
                break;
            case 8: line_pass<8, SIGN, MAXN, NT>(line, p.n, Ns, tw, t); break;
            case 4: line_pass<4, SIGN, MAXN, NT>(line, p.n, Ns, tw, t); break;
            case 2: line_pass<2, SIGN, MAXN, NT>(line, p.n, Ns, tw, t); break;
            case 5: line_pass<5, SIGN, MAXN, NT>(line, p.n, Ns, tw, t); break;
            default: line_pass<3, SIGN, MAXN, NT>(line, p.n, Ns, tw, t); break;
        }
        Ns *= R;
    }
}

}  // namespace dev

// LDS is sized for the next of these lengths.
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

}  // namespace p9idg
