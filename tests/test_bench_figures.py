"""bench.py's byte counts against the passes of the line transforms, counted
array by array, and the rate that it reports for kernels on resampled rows."""
import os
import sys

import numpy as np

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402
import p9idg  # noqa: E402


def test_footprint_and_stage_bytes():
    G, S, L = 96, 8, 3
    meta = np.zeros(4, p9idg.SUBGRID_DTYPE)
    meta["UPixel"] = [10, 30, 40, 20]
    meta["VPixel"] = [12, 12, 50, 20]
    meta["WLambda"] = [0, 0, 1, -1]  # the last mirrors to layer 0
    area, height, width = bench.wstack_footprint(meta, G, S, L)
    # layer 0: (10, 12), (30, 12) and the mirror of (20, 20) at 96 - 20 - 8 + 1 = 69
    assert (area, height, width) == ((69 + 8 - 12) * (69 + 8 - 10) + 8 * 8, 69 + 8 - 12, 69 + 8 - 10)
    got = bench.stage_bytes(G, area, height, width)
    c64, f32 = np.dtype(np.complex64).itemsize, np.dtype(np.float32).itemsize
    box, columns, image = height * width * c64, G * width * c64, G * G * f32
    half, grid = (G // 2 + 1) * G * c64, G * G * c64
    assert got == {"zero": area * c64,
                   "to_image": (area * c64 + box) + (box + columns) + (columns + image),
                   "to_uvw": (image + half) + (half + grid)}


def test_no_fraction_of_a_peak_for_work_that_is_not_done():
    assert bench.direct_sum_tflops(32, 10 ** 6, 1.0) == 8.0 * 1024 * 1e6 / 1e-3 / 1e12
    text = open(bench.__file__).read()
    assert "PEAK_TFLOPS" not in text and text.count("frac") == text.count("frac_of_peak")
