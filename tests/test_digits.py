"""The fixed-point operands of the decode step's integer matrix instructions, compiled for the host."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def weight_digits(tmp_path_factory):
    d = tmp_path_factory.mktemp("digits")
    src, so = str(d / "digits.cpp"), str(d / "digits.so")
    with open(src, "w") as f:
        f.write('#include "cq_digits.h"\nextern "C" void weights(const float* e, float grid, long n, unsigned* o) '
                "{ for (long i = 0; i < n; ++i) o[i] = cq::weight_digits(e[i], grid); }\n")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "calibquant_amd", "csrc"), src, "-o", so], check=True)
    lib = ctypes.CDLL(so)

    def run(e, grid):
        e = np.ascontiguousarray(e, np.float32)
        o = np.empty(e.shape, np.uint32)
        lib.weights(e.ctypes.data_as(ctypes.c_void_p), ctypes.c_float(grid), ctypes.c_long(e.size), o.ctypes.data_as(ctypes.c_void_p))
        d = o[:, None].view(np.int8).reshape(-1, 4).astype(np.int64)
        return d @ (256 ** np.arange(4))
    return run


@pytest.mark.parametrize("grid_bits", [30, 17, 120])
def test_weight_digits_hold_the_nearest_grid_step(weight_digits, grid_bits):
    """A weight is off by half a grid step at most, and not at all where its own last place is a step or more: 24 bits of it
    are kept, as many as it has."""
    rng = np.random.default_rng(3)
    x = np.concatenate([np.exp2(rng.uniform(-12, 30, 200000)), [0.0, 2.0 ** 30, 2.0 ** 23 + 1, 2.0 ** 24 - 1, 2.0 ** 22 + 0.5, 0.5, 1.5]])
    e = (x * 2.0 ** -grid_bits).astype(np.float32)
    steps = e.astype(np.float64) * 2.0 ** grid_bits
    got = weight_digits(e, 2.0 ** grid_bits)
    assert np.abs(got - steps).max() <= 0.5
    assert np.array_equal(got[steps >= 2 ** 23], steps[steps >= 2 ** 23].astype(np.int64))
