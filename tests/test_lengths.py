"""Every fixed transform length on every axis that has it: the device
smoothing filter (an x transform, a y transform in 3-D, a last-axis transform
with a table, and their inverses) against NumPy in double precision.

A single-precision mixed-radix transform of N points has a relative 2-norm
error of about 2^-24 sqrt(log2 N) per direction with rounded twiddles of the
same size; two directions on two or three axes of at most 1024 points stay
below 2e-6 of the largest value for white noise."""

import re
from pathlib import Path

import numpy as np
import pytest

from test_smooth_abi import device_smooth

TEXT = (Path(__file__).parent.parent / "k-wave-ii_amd" / "csrc" / "kw_variants.h").read_text()


def sizes(name):
    start = TEXT.index(f"#define {name}(X)")
    body = TEXT[start:TEXT.index("\n\n", start)]
    return [int(x) for x in re.findall(r"X\((\d+)\)", body)]


ALL, XL = sizes("KW_FIXED_SIZES_ALL"), sizes("KW_FIXED_SIZES_XL")
EMU = sizes("KW_EMU_FIXED_SIZES")


def _check(lib, shape):
    from kwhip.solver import smooth
    f = np.random.default_rng(sum(shape)).standard_normal(shape)
    ref = smooth(f, False)
    err = np.max(np.abs(device_smooth(lib, f) - ref)) / np.max(np.abs(ref))
    assert err <= 2e-6, (shape, err)


def _shapes(n, y):
    return [(n, 15), (15, n)] + ([(8, n, 5)] if y else [])


@pytest.mark.parametrize("n", EMU)
def test_lengths_emu(n):
    from kwhip import _abi
    for shape in _shapes(n, True):
        _check(_abi.load("emu"), shape)


@pytest.mark.gpu
@pytest.mark.parametrize("n", ALL + XL)
def test_lengths_hip(n, hip_lib):
    for shape in _shapes(n, n in ALL):
        _check(hip_lib, shape)


# runtime lengths of x whose threads per pencil are a power of two in small
# launches and the length's own number in these
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(139, 130, 64), (66, 260, 130), (74, 130, 130)])
def test_runtime_lengths_in_large_launches_hip(shape, hip_lib):
    _check(hip_lib, shape)
