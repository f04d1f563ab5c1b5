// Time resampling of the visibilities around the gridder and degridder.
//
// Within a subgrid a baseline's phasor at any pixel (Gridder.cs:62-70),
//   f(t) = exp(2 pi i (off - k (u(t) l + v(t) m + w(t) n))),
// is a smooth function of the timestep: Earth rotation moves the uv point by
// a few hundredths of a grid pixel per step.  Over a chunk of `len` steps it
// therefore equals its Chebyshev interpolant f(t) = sum_j W[t][j] f(t_j) on
// `nodes` < len nodes t_j, with real weights W that depend on (len, nodes)
// only, and the subgrid sums rearrange to
//   gridder:   sum_t V[t] f(t)      = sum_j (sum_t W[t][j] V[t]) f(t_j)
//   degridder: conj f(t) contracted = sum_j W[t][j] (conj f(t_j) contracted)
// so the gridder reads `nodes` rows of channels per chunk instead of `len`,
// and the degridder's rows are interpolated back to the timesteps.
// Observations whose tracks move 0.01-0.1 pixel per step keep 1/6-1/10 of
// their rows.
//
// Which chunks qualify is measured, not assumed: analyse_kernel evaluates the
// interpolant at every timestep of the chunk, at the four corner pixels (where
// the phase varies most) and the highest channel, against the phasor of the
// track itself, from an estimate of the nodes that its phase needs upwards in
// steps of four, and takes the first number whose error is below kResampleTol
// everywhere.  A track with a jump, noise or a gap fails the test and keeps its
// rows as they are.
//
// Long chunks need fewer nodes in all (they grow with the phase that a chunk
// covers, with some ten on top for each), but more weights and products per
// row.  3072^2, subgrid 32, at most 256 / 512 / 1024 timesteps: gridder (two-part
// operands) 141 / 132 / 124 us, gather 45 / 50 / 66; images at 1024^2 with FP32
// 106 / 93 us, three uneven observations 646 / 597.  A chunk that would need more than 64 nodes is
// halved.
#include "device_common.h"

namespace p9idg {
namespace dev {

constexpr int kAnalyse = 256;  // threads of analyse_kernel
constexpr int kMaxNodes = kResampleMaxNodes;
// samples that the track itself is interpolated from (degree 11: exact to
// ~1e-14 of the track for chunks of an hour)
constexpr int kBase = 12;

typedef float rs_f32x4 __attribute__((ext_vector_type(4)));

// Angle of timestep t in an interval of `span` (x = cos(angle) runs from 1 to
// -1) and of Chebyshev node j of J.
__device__ __forceinline__ double angle_of(double t, int span) {
    const double x = 1.0 - 2.0 * t / (double)(span - 1);
    return acos(fmin(1.0, fmax(-1.0, x)));
}
__device__ __forceinline__ double node_angle(int j, int J) { return (kTwoPi / 4.0) * (double)(2 * j + 1) / (double)J; }

// Cardinal function of node j at angle th: with D = th - th_j,
//   w = sin(th_j) sin(J D) / (2 J sin((th + th_j) / 2) sin(D / 2)),
// the Lagrange polynomial of the node written without a difference of cosines.
__device__ __forceinline__ double cardinal(double th, double thj, int J) {
    const double d = th - thj;
    const double ratio = fabs(d) < 1e-12 ? 2.0 * (double)J : sin((double)J * d) / sin(0.5 * d);
    return sin(thj) * ratio / (2.0 * (double)J * sin(0.5 * (th + thj)));
}

// The chunk's base samples: distinct timesteps near Chebyshev nodes.
__device__ __forceinline__ int base_sample(int b, int nb, int len) {
    if (nb >= len) return b;
    const double t = 0.5 * (double)(len - 1) * (1.0 - cos((kTwoPi / 2.0) * (double)b / (double)(nb - 1)));
    int s = (int)rint(t);
    return min(max(s, b), len - nb + b);  // distinct: at least b from either end
}

// The chunk's base samples in LDS: the track there, the timesteps and the
// Lagrange form's constant factors 1 / prod (t_b - t_q), which every node shares.
// All threads of the workgroup.
struct Base {
    double track[kBase][3], t[kBase], inv[kBase];
};
__device__ __forceinline__ void load_base(Base& s, const double* track, int nb, int len) {
    const int tid = threadIdx.x;
    if (tid < nb) {
        const int t = base_sample(tid, nb, len);
        s.t[tid] = (double)t;
        for (int k = 0; k < 3; k++) s.track[tid][k] = track[(size_t)t * 3 + k];
    }
    __syncthreads();
    if (tid < nb) {
        double p = 1.0;
        for (int q = 0; q < nb; q++)
            if (q != tid) p *= s.t[tid] - s.t[q];
        s.inv[tid] = 1.0 / p;
    }
    __syncthreads();
}

// The track at time t from the nb base samples (Lagrange form, FP64).
__device__ __forceinline__ void track_at(double t, const Base& s, int nb, double out[3]) {
    out[0] = out[1] = out[2] = 0.0;
    for (int b = 0; b < nb; b++) {
        double w = s.inv[b];
        for (int q = 0; q < nb; q++)
            if (q != b) w *= t - s.t[q];
        out[0] += w * s.track[b][0];
        out[1] += w * s.track[b][1];
        out[2] += w * s.track[b][2];
    }
}

__device__ __forceinline__ double block_max_d(double v, double* red) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// One workgroup per chunk (thread t: timesteps t, t + 256): a multiple of four
// nodes whose interpolant reproduces the corner phasors of every timestep to
// kResampleTol, or 0: the first that does from an estimate of the phase on.  kl,
// kn: highest wavenumber / 2 pi times the corner pixel's l and n.
//
// The interpolant is evaluated in its barycentric form, with weights (-1)^j
// sin(th_j) / (x - x_j), whose rounding cancels between numerator and denominator:
// a division per timestep and node instead of four sines.  No timestep is a node:
// the timesteps' x are rational, and the rational cosines 0 and 1 / 2 take J = 2 j +
// 1 or 2 J = 3 (2 j + 1), but J is even (an accident of rounding would fail the
// test, no more).  Headline tracks 1040 -> 232 us, 780 baselines x 500 timesteps
// 203 -> 57, 276 x 300 77 -> 35.
__global__ __launch_bounds__(kAnalyse) void analyse_kernel(const ResampleChunk* chunks, const double* uvw, double kl,
                                                           double kn, int32_t* nodes_out) {
    static_assert(kAnalyse == 256, "four waves reduce");
    constexpr int kPer = kResampleMaxLen / kAnalyse;
    __shared__ Base s_base;
    __shared__ double2 s_node[kMaxNodes][4];
    __shared__ double2 s_bary[kMaxNodes];  // x_j and (-1)^j sin(th_j)
    __shared__ double s_red[4];
    const ResampleChunk c = chunks[blockIdx.x];
    const int tid = threadIdx.x, len = c.len, span = c.span;
    const int nb = min(kBase, len);
    const double* track = uvw + (size_t)c.src * 3;
    load_base(s_base, track, nb, len);
    // a timestep's corner phasors relative to the chunk's first sample; the largest phase in turns
    const double u0 = s_base.track[0][0], v0 = s_base.track[0][1], w0 = s_base.track[0][2];
    auto corners = [&](double u, double v, double w, double2* out) {
        const double du = (u - u0) * kl, dv = (v - v0) * kl, dw = (w - w0) * kn;
        double most = 0.0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const double ph = ((q & 1) ? -du : du) + ((q & 2) ? -dv : dv) + dw;
            sincospi(2.0 * ph, &out[q].y, &out[q].x);
            most = fmax(most, fabs(ph));
        }
        // not finite: fails every test below
        return fabs(du) < 1e12 && fabs(dv) < 1e12 && fabs(dw) < 1e12 ? most : 1e9;
    };
    double2 own[kPer][4];
    double x[kPer], phase = 0.0;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int t = tid + k * kAnalyse;
        if (t < len) phase = fmax(phase, corners(track[(size_t)t * 3], track[(size_t)t * 3 + 1], track[(size_t)t * 3 + 2], own[k]));
        x[k] = 1.0 - 2.0 * (double)t / (double)(span - 1);
    }
    // start where the Chebyshev coefficients 2 (z / 2)^J / J! of exp(i z s) fall
    // below the tolerance for z of half the span from the first sample
    phase = block_max_d(phase, s_red);
    const double z = (kTwoPi / 2.0) * phase;
    int start = 1;
    double term = 2.0 * (0.5 * z);
    while (start < kMaxNodes && (term > kResampleTol || (double)start < 0.5 * z)) {
        start++;
        term *= 0.5 * z / (double)start;
    }
    const int limit = min(kMaxNodes, (int)(kResampleKeep * (double)len)) & ~3;
    int found = 0;
    for (int J = (start + 3) & ~3; J <= limit; J += 4) {  // uniform
        __syncthreads();  // the previous candidate's nodes are read
        if (tid < J) {
            double s, co, p[3];
            sincos(node_angle(tid, J), &s, &co);
            s_bary[tid] = make_double2(co, tid & 1 ? -s : s);
            track_at(0.5 * (double)(span - 1) * (1.0 - co), s_base, nb, p);
            double2 n[4];
            corners(p[0], p[1], p[2], n);
#pragma unroll
            for (int q = 0; q < 4; q++) s_node[tid][q] = n[q];
        }
        __syncthreads();
        double err = 0.0;
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            if (tid + k * kAnalyse >= len) continue;
            double den = 0.0;
            double2 num[4] = {};
            for (int j = 0; j < J; j++) {
                const double2 b = s_bary[j];
                const double w = b.y / (x[k] - b.x);
                den += w;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    num[q].x += w * s_node[j][q].x;
                    num[q].y += w * s_node[j][q].y;
                }
            }
            const double inv = 1.0 / den;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const double ex = own[k][q].x - num[q].x * inv, ey = own[k][q].y - num[q].y * inv;
                const double m = fmax(fabs(ex), fabs(ey));
                // fmax passes over a NaN, so both parts are looked at
                err = m <= kResampleTol && ex == ex && ey == ey ? fmax(err, m) : 1e9;
                if (err > kResampleTol) break;
            }
            if (err > kResampleTol) break;
        }
        if (block_max_d(err, s_red) <= kResampleTol) {
            found = J;
            break;
        }
    }
    if (tid == 0) nodes_out[blockIdx.x] = found;
}

// Weights of one (span, nodes) pair per kWeightParts workgroups, FP64 rounded to
// float, in both orders: [t][j] for the degridder's interpolation, [j][t] behind it for
// the gridder's sums.
constexpr int kWeightParts = 16;  // headline tracks: 150 us with one, 51
__global__ void weights_kernel(const ResamplePair* pairs, float* weights) {
    const ResamplePair p = pairs[blockIdx.x / kWeightParts];
    float* tj = weights + p.offset;
    float* jt = tj + (size_t)p.span * p.nodes;
    for (int i = (blockIdx.x % kWeightParts) * blockDim.x + threadIdx.x; i < p.span * p.nodes; i += kWeightParts * blockDim.x) {
        const int t = i / p.nodes, j = i - t * p.nodes;
        const float w = (float)cardinal(angle_of((double)t, p.span), node_angle(j, p.nodes), p.nodes);
        tj[i] = w;
        jt[(size_t)j * p.span + t] = w;
    }
}

// Track rows of the resampled observation: the track at the nodes, or the
// chunk's own rows where it is not resampled.
__global__ __launch_bounds__(kAnalyse) void node_track_kernel(const ResampleChunk* chunks, const double* uvw, double* out) {
    __shared__ Base s_base;
    const ResampleChunk c = chunks[blockIdx.x];
    const int tid = threadIdx.x, nb = min(kBase, c.len);
    const double* track = uvw + (size_t)c.src * 3;
    if (c.nodes == 0) {
        for (int i = tid; i < 3 * c.len; i += blockDim.x) out[(size_t)c.dst * 3 + i] = track[i];
        return;
    }
    load_base(s_base, track, nb, c.len);
    if (tid < c.nodes) {
        double p[3];
        track_at(0.5 * (double)(c.span - 1) * (1.0 - cos(node_angle(tid, c.nodes))), s_base, nb, p);
        for (int k = 0; k < 3; k++) out[((size_t)c.dst + tid) * 3 + k] = p[k];
    }
}

// Four consecutive floats, 4-byte aligned.
__device__ __forceinline__ rs_f32x4 load4(const float* p) {
    rs_f32x4 v;
    __builtin_memcpy(&v, p, sizeof(v));
    return v;
}

// The `count` (even) floats of a chunk that is kept as it is, by wave `w` of
// `waves`, four vectors in flight per lane.
__device__ __forceinline__ void copy_rows(const float* in, float* out, int count, int lane, int w, int waves) {
    constexpr int U = 4;
    const int step = 256 * waves;
    for (int i = (64 * w + lane) * 4; i < count; i += U * step) {
        rs_f32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i + u * step + 3 < count) v[u] = load4(in + i + u * step);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int at = i + u * step;
            if (at + 3 < count)
                __builtin_memcpy(out + at, &v[u], sizeof(v[u]));
            else if (at < count)
                for (int k = 0; k < 2; k++) out[at + k] = in[at + k];
        }
    }
}

// A lane's four neighbouring columns c .. c + 3 of a row of `width` (even).
__device__ __forceinline__ void store4(float* row, int c, int width, rs_f32x4 v) {
    if (c + 3 < width)
        __builtin_memcpy(row + c, &v, sizeof(v));
    else if (c < width)
        __builtin_memcpy(row + c, &v, 2 * sizeof(float));
}

// One chunk's 16 columns for up to 16 Q nodes, in one sweep over the timesteps
// (steps of 16; SPLIT waves take turns), two steps in flight.  MFMA k of a step
// takes timestep 4 g + k from lane group g, so that a lane's four weights of a
// node lie side by side in w[j][t].  sum: LDS of [SPLIT - 1][16][64] floats.
template <int Q, int SPLIT>
__device__ __forceinline__ void gather_chunk(const float* src, const float* w, float* dst, int len, int span, int J,
                                             int width, int n, int nc, int m, int g, int part, float* sum) {
    rs_f32x4 acc[Q];
    const float* row[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        acc[q] = (rs_f32x4){};
        row[q] = w + (size_t)min(16 * q + m, J - 1) * span + 4 * g;
    }
    const int full = len & ~15;
    const float* in = src + (size_t)(4 * g) * width + nc;
    constexpr int D = 2, kStep = 16 * SPLIT;
    float v[D][4];
    rs_f32x4 wt[D][Q];
    auto load = [&](int d, int t0) {
#pragma unroll
        for (int k = 0; k < 4; k++) v[d][k] = in[(size_t)(t0 + k) * width];
#pragma unroll
        for (int q = 0; q < Q; q++) wt[d][q] = load4(row[q] + t0);
    };
#pragma unroll
    for (int d = 0; d < D; d++)
        if (16 * part + kStep * d < full) load(d, 16 * part + kStep * d);
    for (int t1 = 16 * part; t1 < full; t1 += kStep * D)
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int t0 = t1 + kStep * d;
            if (t0 >= full) break;
            float b[4];
            rs_f32x4 a[Q];
#pragma unroll
            for (int k = 0; k < 4; k++) b[k] = v[d][k];
#pragma unroll
            for (int q = 0; q < Q; q++) a[q] = wt[d][q];
            if (t0 + kStep * D < full) load(d, t0 + kStep * D);
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int q = 0; q < Q; q++)
                    acc[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[k], a[q][k], acc[q], 0, 0, 0);
        }
    if (full < len && full / 16 % SPLIT == part) {  // the weights' rows reach to span
        float b[4];
        rs_f32x4 a[Q];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int t = full + 4 * g + k;
            const float x = src[(size_t)min(t, len - 1) * width + nc];
            b[k] = t < len ? x : 0.f;
        }
#pragma unroll
        for (int q = 0; q < Q; q++) a[q] = load4(row[q] + full);
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int q = 0; q < Q; q++) acc[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[k], a[q][k], acc[q], 0, 0, 0);
    }
    if (SPLIT > 1) {
        const int lane = 16 * g + m;
        if (part > 0)
#pragma unroll
            for (int q = 0; q < Q; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) sum[((part - 1) * 16 + 4 * q + r) * 64 + lane] = acc[q][r];
        __syncthreads();
        if (part > 0) return;
#pragma unroll
        for (int p = 0; p < SPLIT - 1; p++)
#pragma unroll
            for (int q = 0; q < Q; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[q][r] += sum[(p * 16 + 4 * q + r) * 64 + lane];
    }
#pragma unroll
    for (int q = 0; q < Q; q++)
        if (16 * q + m < J) store4(dst + (size_t)(16 * q + m) * width, n - m + 4 * g, width, acc[q]);
}

// out[j][n] = sum_t W[t][j] in[t][n] for every chunk, n over the real columns
// of a row of channels, on v_mfma_f32_16x16x4_f32: FP32 products and sums on
// the matrix cores, so the visibilities and weights keep 24 bits.  A wave owns
// a chunk and 16 columns (8 channels); with SPLIT 4 the workgroup's waves share
// them.  Bound by the reads of the visibilities: 134 MB (3072^2) in 37 us, 47
// with one weight per load and one step in flight.
template <int SPLIT>
__global__ __launch_bounds__(256) void gather_rows_kernel(const ResampleChunk* chunks, int nchunks, int ntiles,
                                                          const float* weights, int width, const float* in, float* out) {
    __shared__ float s_sum[SPLIT > 1 ? (SPLIT - 1) * 16 * 64 : 1];
    const int wave = threadIdx.x >> 6, part = SPLIT > 1 ? wave : 0;
    const int unit = SPLIT > 1 ? (int)blockIdx.x : (int)(blockIdx.x * 4 + wave);
    const int ci = unit / ntiles;
    if (ci >= nchunks) return;  // whole waves, or workgroups where they share
    const ResampleChunk c = chunks[ci];
    const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
    const int n = (unit - ci * ntiles) * 16 + m;
    const bool col = n < width;
    const float* src = in + (size_t)c.src * width;
    float* dst = out + (size_t)c.dst * width;
    if (c.nodes == 0) return copy_rows(src, dst, c.len * width, lane, (unit - ci * ntiles) * SPLIT + part, ntiles * SPLIT);
    const int J = c.nodes, len = c.len, nc = col ? n : 0;
    const float* w = weights + c.weights + (size_t)c.span * J;  // [j][t]
    switch ((J + 15) >> 4) {  // uniform
        case 1: return gather_chunk<1, SPLIT>(src, w, dst, len, c.span, J, width, n, nc, m, g, part, s_sum);
        case 2: return gather_chunk<2, SPLIT>(src, w, dst, len, c.span, J, width, n, nc, m, g, part, s_sum);
        case 3: return gather_chunk<3, SPLIT>(src, w, dst, len, c.span, J, width, n, nc, m, g, part, s_sum);
        default: return gather_chunk<4, SPLIT>(src, w, dst, len, c.span, J, width, n, nc, m, g, part, s_sum);
    }
}

// One chunk's 16 columns from up to 16 Q node rows, held in registers, the next
// 16 timesteps' weights in flight (the four waves take turns).  MFMA k of quad q
// takes node 16 q + 4 g + k from lane group g: four weights side by side in
// w[t][j] (J is a multiple of 4).
template <int Q>
__device__ __forceinline__ void spread_chunk(const float* src, const float* w, float* dst, int len, int J, int width, int n,
                                             int nc, int m, int g, int part) {
    float b[Q][4];
    int at[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int j = 16 * q + 4 * g;
        at[q] = min(j, J - 4);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float x = src[(size_t)(at[q] + k) * width + nc];
            b[q][k] = j < J ? x : 0.f;
        }
    }
    rs_f32x4 wt[Q];
    auto load = [&](int t0) {
        const float* row = w + (size_t)min(t0 + m, len - 1) * J;
#pragma unroll
        for (int q = 0; q < Q; q++) wt[q] = load4(row + at[q]);
    };
    load(16 * part);
    for (int t0 = 16 * part; t0 < len; t0 += 64) {
        rs_f32x4 a[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) a[q] = wt[q];
        if (t0 + 64 < len) load(t0 + 64);
        rs_f32x4 acc[2] = {(rs_f32x4){}, (rs_f32x4){}};
#pragma unroll
        for (int q = 0; q < Q; q++)
#pragma unroll
            for (int k = 0; k < 4; k++)
                acc[k & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[q][k], a[q][k], acc[k & 1], 0, 0, 0);
        rs_f32x4 sum;
#pragma unroll
        for (int r = 0; r < 4; r++) sum[r] = acc[0][r] + acc[1][r];
        if (t0 + m < len) store4(dst + (size_t)(t0 + m) * width, n - m + 4 * g, width, sum);
    }
}

// out[t][n] = sum_j W[t][j] in[j][n]: the degridded nodes interpolated to the
// timesteps, 16 timesteps x 16 columns per MFMA tile, a workgroup per chunk and
// 16 columns (one wave each: 46 us at 3072^2).  Bound by the writes: 134 MB
// (3072^2) in 35 us, 50 with one weight per load and one float per store.
__global__ __launch_bounds__(256) void spread_rows_kernel(const ResampleChunk* chunks, int ntiles,
                                                          const float* weights, int width, const float* in, float* out) {
    const int part = threadIdx.x >> 6, unit = blockIdx.x;
    const int ci = unit / ntiles;
    const ResampleChunk c = chunks[ci];
    const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
    const int n = (unit - ci * ntiles) * 16 + m;
    const bool col = n < width;
    const float* src = in + (size_t)c.dst * width;
    float* dst = out + (size_t)c.src * width;
    if (c.nodes == 0) return copy_rows(src, dst, c.len * width, lane, (unit - ci * ntiles) * 4 + part, ntiles * 4);
    const int J = c.nodes, len = c.len, nc = col ? n : 0;
    const float* w = weights + c.weights;  // [t][j]
    switch ((J + 15) >> 4) {  // uniform
        case 1: return spread_chunk<1>(src, w, dst, len, J, width, n, nc, m, g, part);
        case 2: return spread_chunk<2>(src, w, dst, len, J, width, n, nc, m, g, part);
        case 3: return spread_chunk<3>(src, w, dst, len, J, width, n, nc, m, g, part);
        default: return spread_chunk<4>(src, w, dst, len, J, width, n, nc, m, g, part);
    }
}

}  // namespace dev

hipError_t launch_resample_analyse(const ResampleChunk* chunks, int nchunks, const double* uvw, double kl, double kn,
                                   int32_t* nodes, hipStream_t st) {
    if (nchunks <= 0) return hipSuccess;
    hipLaunchKernelGGL(dev::analyse_kernel, dim3(nchunks), dim3(dev::kAnalyse), 0, st, chunks, uvw, kl, kn, nodes);
    return hipGetLastError();
}
hipError_t launch_resample_tables(const ResamplePair* pairs, int npairs, float* weights, const ResampleChunk* chunks,
                                  int nchunks, const double* uvw, double* out, hipStream_t st) {
    if (npairs > 0) {
        hipLaunchKernelGGL(dev::weights_kernel, dim3(npairs * dev::kWeightParts), dim3(256), 0, st, pairs, weights);
        if (hipError_t e = hipGetLastError()) return e;
    }
    if (nchunks > 0)
        hipLaunchKernelGGL(dev::node_track_kernel, dim3(nchunks), dim3(dev::kAnalyse), 0, st, chunks, uvw, out);
    return hipGetLastError();
}
namespace {
// (chunk, column tile) units; below kSplitUnits of them, fewer waves than the
// chip holds, four waves share each in the gather: 1327 units of 256 timesteps
// 11.1 -> 9.5 us; with up to 512, split FP16 at subgrid 64 346 -> 340 us and
// three uneven observations 634 -> 625.
constexpr int64_t kSplitUnits = 8192;
int64_t row_units(int64_t nchunks, int C) { return nchunks * ((2 * C + 15) / 16); }
}  // namespace
bool resample_launches(int64_t nchunks, int C) { return row_units(nchunks, C) <= (int64_t)(UINT32_MAX / 256); }
hipError_t launch_resample_gather(const Resample& r, int C, const float2* vis, float2* out, hipStream_t st) {
    if (r.nchunks <= 0) return hipSuccess;
    const int64_t units = row_units(r.nchunks, C);
    const bool split = units < kSplitUnits;
    hipLaunchKernelGGL(split ? dev::gather_rows_kernel<4> : dev::gather_rows_kernel<1>,
                       dim3((unsigned)(split ? units : (units + 3) / 4)), dim3(256), 0, st, r.chunks, r.nchunks,
                       (2 * C + 15) / 16, r.weights, 2 * C, reinterpret_cast<const float*>(vis),
                       reinterpret_cast<float*>(out));
    return hipGetLastError();
}
hipError_t launch_resample_spread(const Resample& r, int C, const float2* rows, float2* vis, hipStream_t st) {
    if (r.nchunks <= 0) return hipSuccess;
    hipLaunchKernelGGL(dev::spread_rows_kernel, dim3((unsigned)row_units(r.nchunks, C)), dim3(256), 0, st, r.chunks,
                       (2 * C + 15) / 16, r.weights, 2 * C, reinterpret_cast<const float*>(rows),
                       reinterpret_cast<float*>(vis));
    return hipGetLastError();
}

}  // namespace p9idg
