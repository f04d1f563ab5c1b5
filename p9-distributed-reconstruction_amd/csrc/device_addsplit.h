// Adder (scatter of a subgrid onto the grid / w-layers) and splitter
// (gather of a subgrid from the grid), shared by the FP32 and MFMA kernels.
//   Adder.Add        Adder.cs:13-55       AdderWStack.Add    AdderWStack.cs:11-78
//   Adder.Split      Adder.cs:57-95       AdderWStack.Split  AdderWStack.cs:81-139
// The grid is addressed in its FFT.Shift-ed layout (FFT.cs:221-264).
#pragma once

#include "device_common.h"

namespace p9idg {
namespace dev {

// Adds the (normalised) subgrid tile onto the grid.  `tile` is the subgrid
// after the inverse FFT, indexed [y][x] in FFT order.  With a.scratch set the
// values that would be added at grid pixel (Y + y, X + x) are stored at
// scratch[slot][y][x] instead (Y, X: the corner after the negative-w mirror),
// for the ordered sum of gather_slots.  ap: the [S][S] adder phasors
// (a.adder_phasor or a copy of it in LDS).
//
// Thread pairs take the real and the imaginary part of one pixel, so a wave's
// float atomics cover 256 contiguous bytes of a grid row.  The subgrids of the
// short baselines pile up on a few thousand 64-byte sectors (up to ~1000
// subgrids each on the 3072^2 workload) and the adder is bound by the atomics
// that queue on them: a thread per pixel with one atomic per part touches each
// sector twice.  3072^2 gridding of resampled rows 215 -> 186 us.
template <int S>
__device__ __forceinline__ void adder(const KernelArgs& a, const SubgridGeom& g,
                                      const float2* tile, float norm, int slot, const float2* ap) {
    const int G = a.G;
    float* const out = a.scratch ? reinterpret_cast<float*>(a.scratch + (size_t)slot * S * S) : nullptr;
    // Adder.cs:22-47: one grid (range validated on the host: 0 <= U,V < G-S);
    // AdderWStack.cs:29-74: negative w layers are mirrored and conjugated
    const bool plain = a.mode == P9IDG_GRID_PLAIN;
    const bool neg = !plain && g.W < 0;
    int X = g.U, Y = g.V, W = g.W;
    if (neg) {
        X = G - X - S + 1;
        Y = G - Y - S + 1;
        W = -W - 1;
    }
    if (!plain) {
        if (!(X >= 1 && X < G - S && Y >= 1 && Y < G - S)) return;
        if (W < 0 || W >= a.L) return;  // metadata validated on the host
    }
    float* const layer = reinterpret_cast<float*>(a.grid + (a.mode == P9IDG_GRID_WSTACK ? (size_t)W * G * G : 0));
    for (int q = item_tid(); q < 2 * S * S; q += kThreads) {
        const int p = q >> 1, im = q & 1;
        const int y = p / S, x = p - (p / S) * S;
        const int y_ = neg ? S - 1 - y : y;
        const int x_ = neg ? S - 1 - x : x;
        const int ys = (y_ + S / 2) % S, xs = (x_ + S / 2) % S;
        const float2 t = tile[ys * S + xs], f = ap[y_ * S + x_];
        // (im ? Im : Re) of f * t
        const float u = im ? f.y : f.x, w = im ? f.x : -f.y;
        float v = (u * t.x + w * t.y) * norm;
        if (neg && im) v = -v;
        if (out)
            out[q] = v;
        else
            unsafeAtomicAdd(layer + 2 * shift_index(Y + y, X + x, G) + im, v);
    }
}
template <int S>
__device__ __forceinline__ void adder(const KernelArgs& a, const SubgridGeom& g,
                                      const float2* tile, float norm, int slot) {
    adder<S>(a, g, tile, norm, slot, a.adder_phasor);
}

// Reads the subgrid from the model grid into `tile` (FFT order), zeros where
// the reference leaves the subgrid empty.
template <int S>
__device__ __forceinline__ void splitter(const KernelArgs& a, const SubgridGeom& g,
                                         float2* tile) {
    const int G = a.G;
    if (a.mode == P9IDG_DEGRID_PLAIN) {
        // Adder.cs:65-90
        const bool ok = g.U >= 0 && g.U < G - S && g.V >= 0 && g.V < G - S;
        for (int p = item_tid(); p < S * S; p += kThreads) {
            const int y = p / S, x = p - (p / S) * S;
            const int yd = (y + S / 2) % S, xd = (x + S / 2) % S;
            float2 v = make_float2(0.f, 0.f);
            if (ok) {
                float2 gv = a.model_grid[shift_index(g.V + y, g.U + x, G)];
                v = cmulf(gv, conjf2(a.adder_phasor[p]));
            }
            tile[yd * S + xd] = v;
        }
        return;
    }
    // AdderWStack.cs:97-134: one grid; negative w reads the mirrored pixel
    // conjugated; the range test uses the unmirrored corner.
    const bool neg = g.W < 0;
    const int X = g.U, Y = g.V;
    const bool ok = X >= 1 && X < G - S && Y >= 1 && Y < G - S;
    for (int p = item_tid(); p < S * S; p += kThreads) {
        const int y = p / S, x = p - (p / S) * S;
        const int yd = (y + S / 2) % S, xd = (x + S / 2) % S;
        float2 v = make_float2(0.f, 0.f);
        if (ok) {
            const int xs = neg ? G - X - x : X + x;
            const int ys = neg ? G - Y - y : Y + y;
            float2 gv = a.model_grid[shift_index(ys, xs, G)];
            if (neg) gv.y = -gv.y;
            v = cmulf(conjf2(a.adder_phasor[p]), gv);
        }
        tile[yd * S + xd] = v;
    }
}

}  // namespace dev
}  // namespace p9idg
