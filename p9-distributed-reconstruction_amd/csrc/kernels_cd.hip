// Serial coordinate descent (FastSerialCD.cs) and the PSF correlation pieces
// (PaddedConvolver.cs, Common.cs:48-194) on the GPU.
//
// FastSerialCD picks, per iteration, the pixel whose elastic-net proximal
// update changes it most (first row, then first column on ties), writes it
// and adds psf2 * (old - new) to the gradients in the PSF^2 window.  Only the
// window's pixels change, so the argmax is kept as a table of per-tile bests.
// Float expressions use one rounding per operation (no contraction), as the
// reference's float code does (this file is built with -ffp-contract=off).
#include <algorithm>
#include <cmath>

#include "cd_internal.h"

namespace p9idg {
namespace cd {

namespace {

constexpr int kThreads = 256;
constexpr int kSelectThreads = 1024;
constexpr int kDescent = 512;  // threads of a descent workgroup: 3072^2 3.5 us per iteration, 256 3.7, 1024 4.4
constexpr int kCopies = 8;     // of the exchanged words
static_assert(kTile * kTile % kThreads == 0, "whole pixels per thread");

// Common.cs:27-29; Math.Max(v, 0f) gives +0 for -0
__device__ __forceinline__ float prox(float x, float lipschitz, float lambda, float alpha) {
    float num = __fsub_rn(x, __fmul_rn(lambda, alpha));
    num = num > 0.f ? num : 0.f;
    const float den = __fadd_rn(lipschitz, __fmul_rn(lambda, __fsub_rn(1.f, alpha)));
    return __fdiv_rn(num, den);
}

// A candidate update as one ordered word: |old - new| above the complement of
// the pixel index (equal changes: the smaller index wins, as the reference's
// row-then-column scan keeps the first maximum), the sign of old - new in bit
// 0.  0: no update.  Bit 63 is free: a finite or infinite |change| has no sign.
__device__ __forceinline__ Key make_key(float d, int idx) {
    const float m = fabsf(d);
    if (!(m > 0.f)) return 0;
    return ((Key)__float_as_uint(m) << 32) | ((Key)(unsigned)(INT32_MAX - idx) << 1) | (d < 0.f ? 1u : 0u);
}
__device__ __forceinline__ float key_diff(Key k) { return __uint_as_float((unsigned)(k >> 32)); }
__device__ __forceinline__ float key_change(Key k) { return (k & 1) ? -key_diff(k) : key_diff(k); }
__device__ __forceinline__ int key_index(Key k) { return INT32_MAX - (int)((unsigned)k >> 1); }
__device__ __forceinline__ Key max_key(Key a, Key b) { return a > b ? a : b; }

// One step of a wave-wide maximum over DPP lane routes: each lane compares
// with the key CTRL routes to it; lanes outside ROW_MASK (rows of 16 lanes)
// keep their own.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ Key dpp_max(Key k) {
    const int lo = (int)(unsigned)k, hi = (int)(unsigned)(k >> 32);
    const unsigned l = (unsigned)__builtin_amdgcn_update_dpp(lo, lo, CTRL, ROW_MASK, 0xF, false);
    const unsigned h = (unsigned)__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROW_MASK, 0xF, false);
    return max_key(k, ((Key)h << 32) | l);
}
// The wave's largest key, in every lane: lane pairs, quads (quad permutes), 8
// and 16 lanes (half-row and row mirrors), then rows 0 + 1 into row 1 and rows
// 2 + 3 into row 3 (row_bcast15), and rows 0-1 into rows 2-3 (row_bcast31), so
// lane 63 holds the largest of all 64.
__device__ __forceinline__ Key wave_max(Key k) {
    k = dpp_max<0xB1, 0xF>(k);   // quad_perm [1, 0, 3, 2]
    k = dpp_max<0x4E, 0xF>(k);   // quad_perm [2, 3, 0, 1]
    k = dpp_max<0x141, 0xF>(k);  // row_half_mirror
    k = dpp_max<0x140, 0xF>(k);  // row_mirror
    k = dpp_max<0x142, 0xA>(k);  // row_bcast15
    k = dpp_max<0x143, 0xC>(k);  // row_bcast31
    const unsigned l = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)k, 63);
    const unsigned h = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(k >> 32), 63);
    return ((Key)h << 32) | l;
}
template <int WAVES>
__device__ __forceinline__ Key max_of(const Key* v) {
    Key k = v[0];
#pragma unroll
    for (int w = 1; w < WAVES; w++) k = max_key(k, v[w]);
    return k;
}

// FastSerialCD.cs:150-162 for one pixel: the proximal value
__device__ __forceinline__ float update_of(float old, float g, float a, float lambda, float alpha) {
    return prox(__fadd_rn(__fmul_rn(old, a), g), a, lambda, alpha);
}

// What a tile holds besides its best update: whether all its x are +0, and
// whether its Lipschitz values are all `amap`.
struct TileKind {
    float amap;
    bool zero, flat;
};

// The best update of tile (ty, tx), by one wave; own: the tile's gradients
// (p = row * kTile + column), if not NULL.
__device__ __forceinline__ Key tile_best(const float* __restrict__ x, const float* __restrict__ g,
                                         const float* __restrict__ amap, int H, int W, int ty, int tx, float lambda,
                                         float alpha, float* own, TileKind* kind) {
    const int lane = threadIdx.x & 63;
    const int j = tx * kTile + lane % kTile;
    const float first = amap[(size_t)ty * kTile * W + tx * kTile];
    Key best = 0;
    bool zero = true, flat = true;
    if (j < W)
#pragma unroll 8
        for (int r = lane / kTile; r < kTile; r += 64 / kTile) {
            const int i = ty * kTile + r;
            if (i >= H) break;
            const int idx = i * W + j;
            const float old = x[idx], grad = g[idx], a = amap[idx];
            best = max_key(best, make_key(__fsub_rn(old, update_of(old, grad, a, lambda, alpha)), idx));
            if (own) own[r * kTile + lane % kTile] = grad;
            zero = zero && __float_as_uint(old) == 0u;
            flat = flat && __float_as_uint(a) == __float_as_uint(first);
        }
    if (kind) {
        kind->amap = first;
        kind->zero = __all(zero);
        kind->flat = __all(flat);
    }
    return wave_max(best);
}

// One tile per wave.
__global__ __launch_bounds__(kThreads) void tiles_all_kernel(const float* x, const float* g, const float* amap,
                                                             int H, int W, float lambda, float alpha, Key* tiles,
                                                             int ntx, int ntiles) {
    const int t = (int)(blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6));
    if (t >= ntiles) return;
    const Key k = tile_best(x, g, amap, H, W, t / ntx, t % ntx, lambda, alpha, nullptr, nullptr);
    if ((threadIdx.x & 63) == 0) tiles[t] = k;
}

// FastSerialCD.cs:132-135 (GetAbsMaxDiff): the best |diff| of the tile table.
__global__ __launch_bounds__(kSelectThreads) void absmax_kernel(const Key* tiles, int ntiles, State* st) {
    __shared__ Key sh[kSelectThreads / 64];
    Key best = 0;
    for (int i = threadIdx.x; i < ntiles; i += kSelectThreads) best = max_key(best, tiles[i]);
    best = wave_max(best);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) st->absmax = key_diff(max_of<kSelectThreads / 64>(sh));
}

// Common.cs:146-160: flipped PSF at (y + ypad/2 + 1, x + xpad/2 + 1), then
// FFT.Shift (quadrant swap, self-inverse for even N0 = N1)
__global__ void place_correlation_kernel(const float* psf, int ph, int pw, int ypad, int xpad, int N0, int N1,
                                         double2* buf) {
    const size_t n = (size_t)N0 * N1;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int a = (int)(i / N1), b = (int)(i % N1);
        const int h = N0 / 2;
        // quadrant swap of the first h x h block pairs (FFT.cs:248-264)
        int p = a, q = b;
        if (a < 2 * h && b < 2 * h) {
            p = a < h ? a + h : a - h;
            q = b < h ? b + h : b - h;
        }
        const int y = p - ypad / 2 - 1, x = q - xpad / 2 - 1;
        double v = 0.0;
        if (y >= 0 && y < ph && x >= 0 && x < pw) v = (double)psf[(ph - y - 1) * pw + (pw - x - 1)];
        buf[i] = make_double2(v, 0.0);
    }
}

// Common.cs:164-172 (SetPsfInWindow): psf at (i + ph/2, j + pw/2)
__global__ void place_centered_kernel(const float* psf, int ph, int pw, int N0, int N1, double2* buf) {
    const size_t n = (size_t)N0 * N1;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int y = (int)(i / N1) - ph / 2, x = (int)(i % N1) - pw / 2;
        const double v = (y >= 0 && y < ph && x >= 0 && x < pw) ? (double)psf[y * pw + x] : 0.0;
        buf[i] = make_double2(v, 0.0);
    }
}

// PaddedConvolver.cs:95-114
__global__ void insert_image_kernel(const float* img, int H, int W, int yh, int xh, int N0, int N1, double2* buf) {
    const size_t n = (size_t)N0 * N1;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int y = (int)(i / N1) - yh, x = (int)(i % N1) - xh;
        const double v = (y >= 0 && y < H && x >= 0 && x < W) ? (double)img[(size_t)y * W + x] : 0.0;
        buf[i] = make_double2(v, 0.0);
    }
}

__global__ void multiply_kernel(double2* buf, const double2* k, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const double2 a = buf[i], b = k[i];
        buf[i] = make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
    }
}

// PaddedConvolver.cs:58-64
__global__ void extract_kernel(const double2* buf, int N1, int yh, int xh, double norm, int H, int W, float* out) {
    const size_t n = (size_t)H * W;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int y = (int)(i / W), x = (int)(i % W);
        out[i] = (float)(buf[(size_t)(y + yh) * N1 + (x + xh)].x / norm);
    }
}

// Common.cs:88-126 (QueryScan) on the prefix sums of psf^2
__global__ void amap_kernel(const double* s, int ph, int pw, int H, int W, float* amap) {
    const size_t n = (size_t)H * W;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int y = (int)(i / W), x = (int)(i % W);
        const int y_over = max(0, y + (ph - ph / 2) - H), x_over = max(0, x + (pw - pw / 2) - W);
        const int y_under = -(y - ph / 2), x_under = -(x - pw / 2);
        const int yu = max(1, y_under) - 1, xu = max(1, x_under) - 1;
        auto S = [&](int a, int b) { return s[a * pw + b]; };
        double v;
        if (y_over <= 0 && x_over <= 0 && y_under <= 0 && x_under <= 0) {
            v = S(ph - 1, pw - 1);
        } else if (y_under > 0 && x_under > 0) {
            v = S(ph - 1, pw - 1) - S(ph - 1, xu) - S(yu, pw - 1) + S(yu, xu);
        } else {
            double corr = 0.0;
            if (y_under > 0) corr += S(yu, pw - x_over - 1);
            if (x_under > 0) corr += S(ph - y_over - 1, xu);
            v = S(ph - 1 - y_over, pw - 1 - x_over) - corr;
        }
        amap[i] = (float)v;
    }
}

// --- the descent ----------------------------------------------------------------
// All iterations of a call in one cooperative launch.  Tile (ty, tx) belongs to
// workgroup (ty % OH, tx % OW) of an OH x OW arrangement, so the tiles of a
// window fall on different workgroups, and each workgroup keeps the bests of
// its tiles.  An iteration is one exchange: every workgroup publishes its best
// update, reads all of them and finds the same maximum; the owners of the
// window's tiles then add psf2 * (old - new) to their gradients
// (FastSerialCD.cs:219-238) and re-evaluate them.  A pixel is only ever touched
// by one thread of its tile's workgroup.
//
// What bounds it is latency: 2 to 2.6 us of an iteration are the exchange over
// the XCDs, the rest are the window's loads.  A launch pair per iteration
// (window, then a one-workgroup selection) took 9.7 us, most of it between the
// launches.  3072^2, PSF 192^2, 3000 iterations: 29.2 -> 10.5 ms.
//
// A published word holds the key and, in bit 63, the turn's tag, so one 64-bit
// store hands over both and nothing else needs ordering.  Turn n uses buffer
// n & 1 with tag (n >> 1) & 1: a workgroup writes turn n + 2 only after it has
// read turn n + 1 from all, each of which had then finished reading turn n.
// Every buffer has kCopies copies, each polled by every kCopies-th workgroup
// (one copy: 3.3 us per exchange of 256 workgroups instead of 2.6).
//
// RES: the tiles' gradients stay in LDS between the first and the last turn.
// x and the Lipschitz map are read only where a tile's are not all zero or all
// equal, so that a window's tile usually waits for nothing but psf2 (16.5 ->
// 11.1 ms together with the copies).
struct Descent {
    float* x;
    float* g;
    const float* amap;
    const float* psf2;
    int p2h, p2w, H, W, OH, OW;
    float lambda, alpha, epsilon;
    int limit;    // updates of this launch
    Key* slots;   // [2][kCopies][OH * OW], then the gate's two words
    Key* tiles;   // [OH * OW][local]: the tile tables where they don't fit LDS
    int local;
    State* st;
};
constexpr int kLdsTiles = 1024;
constexpr int kResTiles = 38;  // 4 KB each
constexpr Key kStalled = ~(Key)0;
// Polls of the gate: a fraction of a second for the form that wants every CU's
// LDS for itself, after which the one that shares the CUs is tried; that one waits
// longer, as other programs' kernels may hold them, and gives way to one workgroup.
constexpr int kGatePollsRes = 1 << 19, kGatePolls = 1 << 25;
constexpr int kMaxPolls = 1 << 28;

// The slots' tags before turn 0 (neither buffer holds its first turn) and the
// gate: arrivals, verdict.
__global__ void reset_slots_kernel(Key* slots, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n + 2) slots[i] = i < n ? (Key)1 << 63 : 0;
}

__device__ __forceinline__ Key poll(const Key* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ Key await_slot(const Key* slot, unsigned tag) {
    for (int i = 0; i < kMaxPolls; i++) {
        const Key v = poll(slot);
        if ((unsigned)(v >> 63) == tag) return v & ~((Key)1 << 63);
    }
    return kStalled;
}
// Whether all workgroups of the launch are resident: the last to arrive opens
// the gate, the first to lose patience shuts it, and the first verdict holds
// for all.  Nothing has been changed before it.
__device__ __forceinline__ bool all_resident(Key* gate, Key nwg, int polls) {
    if (__hip_atomic_fetch_add(gate, (Key)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == nwg) atomicCAS(gate + 1, (Key)0, (Key)1);
    for (int i = 0; i < polls; i++)
        if (const Key v = poll(gate + 1)) return v == 1;
    const Key before = atomicCAS(gate + 1, (Key)0, (Key)2);
    return before == 1;
}

template <bool LDS, bool RES>
__global__ __launch_bounds__(kDescent) void descent_kernel(Descent a) {
    static_assert(LDS || !RES, "resident tiles have their table in LDS");
    constexpr int kWaves = kDescent / 64, kPer = kTile * kTile / kDescent, kTiles = RES ? kResTiles : LDS ? kLdsTiles : 1;
    __shared__ float s_g[RES ? kResTiles * kTile * kTile : 1];
    __shared__ Key s_table[kTiles];
    __shared__ float s_amap[kTiles];
    __shared__ unsigned char s_zero[kTiles], s_flat[kTiles];
    __shared__ Key s_turn[2][kWaves], s_tile[2][kWaves];
    __shared__ int s_go;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int H = a.H, W = a.W, OH = a.OH, OW = a.OW, me = blockIdx.x, nwg = OH * OW;
    if (t == 0) s_go = all_resident(a.slots + 2 * kCopies * nwg, nwg, RES ? kGatePollsRes : kGatePolls);
    const int ntx = (W + kTile - 1) / kTile, nty = (H + kTile - 1) / kTile;
    const int oy = me / OW, ox = me - oy * OW;
    const int nrow = (nty - oy + OH - 1) / OH, ncol = (ntx - ox + OW - 1) / OW, nlocal = nrow * ncol;
    Key* const table = LDS ? s_table : a.tiles + (size_t)me * a.local;
    for (int l = wave; l < nlocal; l += kWaves) {
        TileKind kind;
        const Key k = tile_best(a.x, a.g, a.amap, H, W, oy + l / ncol * OH, ox + l % ncol * OW, a.lambda, a.alpha,
                                RES ? s_g + l * kTile * kTile : nullptr, LDS ? &kind : nullptr);
        if (lane == 0) {
            table[l] = k;
            if (LDS) {
                s_amap[l] = kind.amap;
                s_zero[l] = kind.zero;
                s_flat[l] = kind.flat;
            }
        }
    }
    __threadfence_block();
    __syncthreads();
    if (!s_go) {
        if (me == 0 && t == 0) a.st->stalled = 1;
        return;  // every workgroup
    }
    const int yh = a.p2h / 2, xh = a.p2w / 2;
    Key mine = 0, best = 0;
    bool changed = true;  // of this workgroup's tiles
    int updates = 0;
    for (unsigned turn = 0;; turn++) {
        Key* const slots = a.slots + (turn & 1) * kCopies * nwg;
        const unsigned tag = (turn >> 1) & 1;
        if (wave == 0) {
            if (changed) {
                mine = 0;
                for (int l = lane; l < nlocal; l += 64) mine = max_key(mine, table[l]);
                mine = wave_max(mine);
            }
            if (lane < kCopies)
                __hip_atomic_store(slots + lane * nwg + me, mine | ((Key)tag << 63), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        Key v = 0;
        for (int s = t; s < nwg; s += kDescent) v = max_key(v, await_slot(slots + me % kCopies * nwg + s, tag));
        v = wave_max(v);
        if (lane == 0) s_turn[turn & 1][wave] = v;
        __syncthreads();
        best = max_of<kWaves>(s_turn[turn & 1]);
        // FastSerialCD.cs:84-97
        if (best == kStalled || best == 0 || key_diff(best) < a.epsilon) break;
        updates++;
        const int at = key_index(best), y0 = at / W, x0 = at - y0 * W;
        const float d = key_change(best);
        const int r0 = max(y0 - yh, 0), r1 = min(y0 - yh + a.p2h, H);
        const int c0 = max(x0 - xh, 0), c1 = min(x0 - xh + a.p2w, W);
        const int tya = r0 / kTile, txa = c0 / kTile, tyb = (r1 - 1) / kTile, txb = (c1 - 1) / kTile;
        int q = 0;
        // the first own tile at or after (tya, txa) in each direction
        for (int ty = tya + (oy + OH - tya % OH) % OH; ty <= tyb; ty += OH)
            for (int tx = txa + (ox + OW - txa % OW) % OW; tx <= txb; tx += OW, q++) {
                const int l = (ty / OH) * ncol + tx / OW;
                const bool zero = LDS && s_zero[l], flat = LDS && s_flat[l];  // uniform but for the update's own clearing of zero
                const float amap = LDS ? s_amap[l] : 0.f;
                int idx[kPer];
                bool in[kPer], win[kPer];
                float gv[kPer], pv[kPer], xv[kPer], av[kPer];
#pragma unroll
                for (int k = 0; k < kPer; k++) {
                    const int p = t + k * kDescent, i = ty * kTile + p / kTile, j = tx * kTile + p % kTile;
                    in[k] = i < H && j < W;
                    win[k] = in[k] && i >= r0 && i < r1 && j >= c0 && j < c1;
                    idx[k] = in[k] ? i * W + j : 0;
                    pv[k] = win[k] ? a.psf2[(i - y0 + yh) * a.p2w + (j - x0 + xh)] : 0.f;
                    gv[k] = RES ? s_g[l * kTile * kTile + p] : in[k] ? a.g[idx[k]] : 0.f;
                    xv[k] = !zero && in[k] ? a.x[idx[k]] : 0.f;
                    av[k] = flat ? amap : in[k] ? a.amap[idx[k]] : 0.f;
                }
                Key b = 0;
#pragma unroll
                for (int k = 0; k < kPer; k++) {
                    if (!in[k]) continue;
                    if (idx[k] == at) {  // the update itself
                        xv[k] = update_of(xv[k], gv[k], av[k], a.lambda, a.alpha);
                        a.x[at] = xv[k];
                        if (LDS) s_zero[l] = 0;
                    }
                    if (win[k]) {
                        gv[k] = __fadd_rn(gv[k], __fmul_rn(pv[k], d));
                        if (RES)
                            s_g[l * kTile * kTile + t + k * kDescent] = gv[k];
                        else
                            a.g[idx[k]] = gv[k];
                    }
                    b = max_key(b, make_key(__fsub_rn(xv[k], update_of(xv[k], gv[k], av[k], a.lambda, a.alpha)), idx[k]));
                }
                b = wave_max(b);
                if (lane == 0) s_tile[q & 1][wave] = b;
                __syncthreads();
                if (t == 0) table[l] = max_of<kWaves>(s_tile[q & 1]);
            }
        changed = q > 0;
        if (changed) __threadfence_block();  // wave 0 reads what its lane 0 wrote
        if (updates >= a.limit) break;
    }
    if (RES)
        for (int l = 0; l < nlocal; l++)
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                const int p = t + k * kDescent;  // this thread's own elements, after a barrier in any case
                const int i = (oy + l / ncol * OH) * kTile + p / kTile, j = (ox + l % ncol * OW) * kTile + p % kTile;
                if (i < H && j < W) a.g[i * W + j] = s_g[l * kTile * kTile + p];
            }
    if (me == 0 && t == 0) {
        const bool stop = updates < a.limit || best == 0 || key_diff(best) < a.epsilon;
        a.st->stalled = best == kStalled ? 2 : 0;
        a.st->updates = updates;
        a.st->done = stop;
        a.st->converged = stop && key_diff(best) < a.epsilon;
    }
}

__global__ void zero_u32_kernel(unsigned* p) { *p = 0u; }

// Residuals.GetMax (Common.cs:244-251): max(0, v) as unsigned bits
__global__ void get_max_kernel(const float* v, size_t n, unsigned* out) {
    float m = 0.f;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        m = fmaxf(m, v[i]);
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) atomicMax(out, __float_as_uint(m));
}

unsigned blocks(size_t n) {
    const size_t b = (n + kThreads - 1) / kThreads;
    return (unsigned)(b > 4096 ? 4096 : (b == 0 ? 1 : b));
}

}  // namespace

hipError_t launch_tiles_all(const float* x, const float* g, const float* amap, int H, int W, float lambda,
                            float alpha, Key* tiles, hipStream_t st) {
    const int ntx = (W + kTile - 1) / kTile, n = ntx * ((H + kTile - 1) / kTile);
    hipLaunchKernelGGL(tiles_all_kernel, dim3((n + kThreads / 64 - 1) / (kThreads / 64)), dim3(kThreads), 0, st, x, g, amap,
                       H, W, lambda, alpha, tiles, ntx, n);
    return hipGetLastError();
}

hipError_t launch_absmax(const Key* tiles, int ntiles, State* state, hipStream_t st) {
    hipLaunchKernelGGL(absmax_kernel, dim3(1), dim3(kSelectThreads), 0, st, tiles, ntiles, state);
    return hipGetLastError();
}

hipError_t launch_place_correlation(const float* psf, int ph, int pw, int ypad, int xpad, int N0, int N1,
                                    double2* buf, hipStream_t st) {
    hipLaunchKernelGGL(place_correlation_kernel, dim3(blocks((size_t)N0 * N1)), dim3(kThreads), 0, st, psf, ph, pw,
                       ypad, xpad, N0, N1, buf);
    return hipGetLastError();
}

hipError_t launch_place_centered(const float* psf, int ph, int pw, int N0, int N1, double2* buf, hipStream_t st) {
    hipLaunchKernelGGL(place_centered_kernel, dim3(blocks((size_t)N0 * N1)), dim3(kThreads), 0, st, psf, ph, pw, N0,
                       N1, buf);
    return hipGetLastError();
}

hipError_t launch_insert_image(const float* img, int H, int W, int yh, int xh, int N0, int N1, double2* buf,
                               hipStream_t st) {
    hipLaunchKernelGGL(insert_image_kernel, dim3(blocks((size_t)N0 * N1)), dim3(kThreads), 0, st, img, H, W, yh, xh,
                       N0, N1, buf);
    return hipGetLastError();
}

hipError_t launch_multiply(double2* buf, const double2* kernel, size_t n, hipStream_t st) {
    hipLaunchKernelGGL(multiply_kernel, dim3(blocks(n)), dim3(kThreads), 0, st, buf, kernel, n);
    return hipGetLastError();
}

hipError_t launch_extract(const double2* buf, int N1, int yh, int xh, double norm, int H, int W, float* out,
                          hipStream_t st) {
    hipLaunchKernelGGL(extract_kernel, dim3(blocks((size_t)H * W)), dim3(kThreads), 0, st, buf, N1, yh, xh, norm, H,
                       W, out);
    return hipGetLastError();
}

namespace {

const void* descent_of(int local, bool resident) {
    return resident && local <= kResTiles ? reinterpret_cast<const void*>(descent_kernel<true, true>)
           : local <= kLdsTiles           ? reinterpret_cast<const void*>(descent_kernel<true, false>)
                                          : reinterpret_cast<const void*>(descent_kernel<false, false>);
}

}  // namespace

hipError_t descent_shape(int H, int W, int p2h, int p2w, DescentShape* shape) {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    const int ntx = (W + kTile - 1) / kTile, nty = (H + kTile - 1) / kTile;
    auto arrange = [&](int side) {
        shape->OW = std::min(side, ntx);
        shape->OH = std::min(nty, side * side / shape->OW);
        shape->OW = std::min(ntx, side * side / shape->OH);
        shape->local = ((nty + shape->OH - 1) / shape->OH) * ((ntx + shape->OW - 1) / shape->OW);
    };
    // The exchange is faster among fewer workgroups, so no more than the
    // window's tiles, unless only more of them hold all gradients in LDS.  us
    // per iteration, 8 x 8 / 11 x 11 / 16 x 16: 512^2 with a 64^2 window 3.1 /
    // 3.3 / 3.8, 1500^2 with 200^2 3.3 / 3.5 / 3.8, 3072^2 with 384^2 (too
    // large for LDS below 16 x 16) 6.3 / 6.4 / 3.5.
    const int most = std::max(1, (int)std::sqrt((double)std::max(cus, 1)));  // one workgroup per CU at most
    const int window = std::max(p2h, p2w) / kTile + 1;
    arrange(std::min(most, std::max(8, window)));
    if (shape->local > kResTiles) arrange(most);
    return hipSuccess;
}

DescentForm descent_form(const DescentShape& shape) { return shape.local <= kResTiles ? kResident : kShared; }

size_t descent_slots(const DescentShape& shape) { return 2 * kCopies * (size_t)shape.OH * shape.OW + 2; }

hipError_t launch_descent(float* x, float* g, const float* amap, const float* psf2, int p2h, int p2w, int H, int W,
                          const DescentShape& shape, DescentForm form, float lambda, float alpha, float epsilon, int limit,
                          Key* slots, Key* tiles, State* state, hipStream_t st) {
    DescentShape sh = shape;
    if (form == kSingle) sh = {1, 1, ((H + kTile - 1) / kTile) * ((W + kTile - 1) / kTile)};
    const int n = sh.OH * sh.OW, words = 2 * kCopies * n;
    hipLaunchKernelGGL(reset_slots_kernel, dim3((words + 2 + kThreads - 1) / kThreads), dim3(kThreads), 0, st, slots, words);
    if (hipError_t e = hipGetLastError()) return e;
    Descent a{x, g, amap, psf2, p2h, p2w, H, W, sh.OH, sh.OW, lambda, alpha, epsilon, limit, slots, tiles, sh.local, state};
    void* args[] = {&a};
    return hipLaunchCooperativeKernel(descent_of(sh.local, form == kResident), dim3(n), dim3(kDescent), args, 0, st);
}

hipError_t launch_amap(const double* scan, int ph, int pw, int H, int W, float* amap, hipStream_t st) {
    hipLaunchKernelGGL(amap_kernel, dim3(blocks((size_t)H * W)), dim3(kThreads), 0, st, scan, ph, pw, H, W, amap);
    return hipGetLastError();
}

hipError_t launch_get_max(const float* v, size_t n, float* out, hipStream_t st) {
    unsigned* o = reinterpret_cast<unsigned*>(out);
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, st, o);
    hipLaunchKernelGGL(get_max_kernel, dim3(blocks(n)), dim3(kThreads), 0, st, v, n, o);
    return hipGetLastError();
}

}  // namespace cd
}  // namespace p9idg
