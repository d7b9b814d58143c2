"""The launch shape a solver starts with: 64-thread workgroups while the
planes do not exceed the SIMDs or the state stays in cache, 128 threads
beyond.  A shape only orders the planes, so every one gives the same bits.
"""
import numpy as np
import pytest

from hemelb_amd import workloads as W

pytestmark = pytest.mark.gpu


# 64 planes, 864 planes, above one plane per SIMD, and above 64 MB of binary32
@pytest.mark.parametrize("radius,length,storage,threads,remap", [
    (5.0, 16, "fp64", 64, 16), (12.0, 96, "fp64", 64, 16), (12.0, 96, "fp32", 64, 16),
    (18.0, 96, "fp64", 64, 0), (18.0, 96, "fp32", 64, 0), (18.0, 96, "fp16", 64, 16),
    (32.0, 192, "fp64", 64, 0), (32.0, 192, "fp32", 128, 8),
])
def test_default_shape_gives_the_same_bits(radius, length, storage, threads, remap):
    w = W.small_cylinder(radius, length)
    print(f"[launch] n={w.domain.n} {storage}", flush=True)
    a, b = w.solver(storage), w.solver(storage)
    shape = a.launch_shape
    assert (shape["threads"], shape["xcd_remap"]) == (threads, remap)
    b.set_launch_shape(threads=256)
    for n in (1, 7):
        a.step(n)
        b.step(n)
        np.testing.assert_array_equal(a.get_distributions(), b.get_distributions())


def test_default_shape_beyond_the_cache_gives_the_same_bits():
    # binary64 above 256 MB of state (1.118 M D3Q15 sites): the shape of the
    # largest domains
    w = W.small_cylinder(40.0, 240)
    print(f"[launch] n={w.domain.n} fp64", flush=True)
    assert 2 * 8 * 15 * w.domain.n > 256 << 20
    a, b = w.solver("fp64"), w.solver("fp64")
    shape = a.launch_shape
    assert (shape["threads"], shape["xcd_remap"]) == (128, 2)
    b.set_launch_shape(threads=256)
    for n in (1, 7):
        a.step(n)
        b.step(n)
        np.testing.assert_array_equal(a.get_distributions(), b.get_distributions())
