"""What two bf16 values miss of an fp32 number: the constants of the bf16 pre-selection's error bound
(vsag_amd/csrc/prefilter_b16.hip) against the split itself, on random floats and at the worst places of the rounding."""
import os
import re

import numpy as np

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vsag_amd", "csrc", "prefilter_b16.hip")


def bf16(x):
    """The nearest bf16 value, ties to even."""
    u = x.view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)


def constant(name):
    with open(SOURCE) as f:
        return float(re.search(r"constexpr double %s = ([0-9.e+-]+);" % name, f.read()).group(1))


def test_constants_cover_the_split():
    rng = np.random.default_rng(1)
    x = np.concatenate([rng.random(1 << 20, dtype=np.float32) + np.float32(1), rng.standard_normal(1 << 20).astype(np.float32),
                        (1 + np.arange(1 << 16) * 2.0 ** -23).astype(np.float32),
                        (1 + (128 + np.arange(-4096, 4096)) * 2.0 ** -16).astype(np.float32)])
    x = x[np.abs(x) > 1e-30]
    high = bf16(x)
    low = bf16(x - high)
    size = np.abs(x.astype(np.float64))
    most_low = np.max(np.abs(low) / size)
    most_left = np.max(np.abs(x.astype(np.float64) - high - low) / size)
    assert 2.0 ** -8 * 0.99 < most_low <= constant("kB16Low")      # the worst case is among the numbers, and covered
    assert 2.0 ** -17 * 0.99 < most_left <= constant("kB16Left")
