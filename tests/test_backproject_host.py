"""Host-side functions of the backprojection: the number of parts that a block's
angles are summed in, and the weight that its kernels evaluate (the same source,
built for the host)."""
import ctypes as C

import numpy as np
import pytest

import ctbangbang_amd as cb


def _function(name, result, *arguments):
    f = getattr(cb.lib(), name)
    f.restype, f.argtypes = result, list(arguments)
    return f


@pytest.mark.parametrize("lo,hi", [(0.0, 0.6), (0.6, 0.9), (0.9, 0.99), (0.99, 0.999), (0.999, 0.9999), (0.9999, 1.0)])
def test_stierstorfer_weight(lo, hi):
    """W(|q|) against 64 bits of t rounded to FP32 (the kernel's input to the
    weight), as a fraction of W up to the edge.  Tolerance 1e-6: the cosine's
    polynomial 2.4e-7, the roundings of v, of P's outer terms and of the sum
    2.3e-7, twice both for the square, and the square's own."""
    weight = _function("_ZN4ctbb18backproject_weightEf", C.c_float, C.c_float)
    q = (lo + (hi - lo) * np.random.default_rng(int(1e4 * hi)).random(20000)).astype(np.float32)
    q = np.unique(np.append(q, np.nextafter(np.float32(hi), np.float32(0))))
    q = q[q < 1]
    got = np.array([weight(float(x)) for x in q])
    t = np.clip((2.5 * q.astype(np.float64) - 1.5).astype(np.float32), 0.0, 1.0)
    want = np.cos(np.float64(np.float32(3.1415368979)) / 2 * t.astype(np.float64)) ** 2
    assert (got > 0).all()
    assert np.abs(got / want - 1).max() <= 1e-6
    if hi <= 0.6:
        assert (got == 1).all()


@pytest.mark.parametrize("n_tiles,half,want", [
    (1024, 576, 1), (512, 576, 1), (4096, 576, 1),              # whole rounds of two workgroups per CU
    (256, 63, 1), (1, 32, 1),                                    # fewer than 32 angles for each part
    (256, 576, 2), (625, 576, 4), (225, 576, 9),
    (32, 512, 16), (1, 4096, 16), (32, 511, 15)])                # the upper limit
def test_backproject_parts_rule(n_tiles, half, want):
    """Parts for 256 compute units: one where the tiles fill whole rounds, never
    more than 16 or than leave 32 angles each."""
    parts = _function("_ZN4ctbb17backproject_partsEiii", C.c_int, C.c_int, C.c_int, C.c_int)
    assert parts(n_tiles, half, 256) == want


@pytest.mark.parametrize("tiles", [1, 6, 40, 272])
def test_backproject_parts_of_small_images(tiles):
    """The images of 16^2 to 272 x 256 with 96 angles that the GPU tests take for
    blocks in parts are."""
    parts = _function("_ZN4ctbb17backproject_partsEiii", C.c_int, C.c_int, C.c_int, C.c_int)
    assert parts(tiles, 96, 256) > 1
