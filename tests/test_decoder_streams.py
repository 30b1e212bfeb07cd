"""Decoders on arbitrary streams, and 4D blocks over four lanes.

Every bit string is a valid fixed-rate stream, so random words drive the plane
decoders where smooth fields seldom do: scans that run past the 64-bit window
of the group tests, scans that the budget or the last coefficient ends, planes
cut inside their verbatim bits, blocks of zeros.  Words of few one-bits give
long runs (up to a whole 4D plane), words of few zero-bits give dense planes.
The codec is integer and exact: every value must equal the oracle's.

4D fields lie at the edges of the four-lane kernels: 16 blocks per coding
wave, 64 per parsing wave, and blocks so long that a wave parses them in
several passes."""
import ctypes
import zlib

import numpy as np
import pytest

from test_device_code_on_host import lib
from zfptest import (NP_OF_TYPE, T_DOUBLE, T_FLOAT, T_INT32, T_INT64, field_args, make_layout, oracle_decompress,
                     pdp, smooth_field, stream_params_accuracy, stream_params_precision, stream_params_rate, szp, u64p)

TYPES = {"i32": T_INT32, "i64": T_INT64, "f32": T_FLOAT, "f64": T_DOUBLE}
DENSITY = {"sparse": 0.01, "even": 0.5, "dense": 0.97}
SHAPES = {"1d": [70], "2d": [13, 21], "3d": [9, 10, 14], "4d": [5, 6, 9, 21]}


def random_stream(n, ztype, rate, density):
    """Random words for a fixed-rate field of extents n, its parameters and its oracle reconstruction."""
    rng = np.random.default_rng(zlib.crc32(f"{n}/{ztype}/{rate}/{density}".encode()))
    params = stream_params_rate(rate, ztype, len(n))
    blocks = int(np.prod([(v + 3) // 4 for v in n]))
    count = (blocks * params[1] + 63) // 64
    bits = rng.random((count, 64)) < DENSITY[density]
    words = np.packbits(bits, axis=1, bitorder="little").view(np.uint64).reshape(-1).copy()
    want = np.zeros(int(np.prod(n)), NP_OF_TYPE[ztype])
    _, off, s = make_layout(want, n, "as_is")
    oracle_decompress(words, want, off, n, s, ztype, params)
    return words, params, want


@pytest.mark.parametrize("density", list(DENSITY))
@pytest.mark.parametrize("rate", [3, 8, 21])
@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("shape", ["1d", "2d", "3d"])
def test_random_streams_host(shape, tname, rate, density):
    n, ztype = SHAPES[shape], TYPES[tname]
    words, params, want = random_stream(n, ztype, rate, density)
    got = np.zeros_like(want)
    nn, ss = field_args(n, None)
    lib().hostcodec_decompress(ztype, nn, ss, got.ctypes.data, *params, words.ctypes.data_as(u64p), words.size, 0)
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    slot = np.zeros_like(want)
    fn = lib().hostcodec_decompress_slot
    fn.restype = ctypes.c_uint64
    fn.argtypes = [ctypes.c_int, szp, pdp, ctypes.c_void_p, ctypes.c_uint, ctypes.c_uint, ctypes.c_int, u64p,
                   ctypes.c_uint64, ctypes.c_uint64]
    fn(ztype, nn, ss, slot.ctypes.data, params[1], params[2], params[3], words.ctypes.data_as(u64p), words.size, 0)
    assert np.array_equal(slot.view(np.uint8), want.view(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("density", list(DENSITY))
@pytest.mark.parametrize("rate", [3, 8, 21])
@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("shape", list(SHAPES))
def test_random_streams_gpu(shape, tname, rate, density):
    import torch

    import zfp_amd as Z
    n, ztype = SHAPES[shape], TYPES[tname]
    words, params, want = random_stream(n, ztype, rate, density)
    w = torch.from_numpy(words.view(np.int64)).cuda()
    out = torch.zeros(want.nbytes, dtype=torch.uint8, device="cuda")
    Z.decode(ztype, n, None, out.data_ptr(), params, w.data_ptr(), nwords=w.numel())
    assert np.array_equal(out.cpu().numpy(), want.view(np.uint8))


MODES_4D = {
    "prec3": lambda t: stream_params_precision(3),
    "prec33": lambda t: stream_params_precision(33),   # the low half's first plane
    "prec64": lambda t: stream_params_precision(64),   # the longest blocks
    "acc1e-4": lambda t: stream_params_accuracy(1e-4),
    "expert": lambda t: (700, 3000, 40, -40),          # padding and a budget
}


def field_4d(n, ztype, content):
    if content == "smooth":
        return smooth_field(n, ztype, seed=sum(n))
    rng = np.random.default_rng(sum(n))
    count = int(np.prod(n))
    a = np.zeros(count, NP_OF_TYPE[ztype])
    if content == "noise":
        a[:] = (rng.random(count) * 2 - 1) * (2.0 ** 28 if ztype in (T_INT32, T_INT64) else 1.0)
    else:
        # whole blocks of zeros beside single values
        pick = rng.random(count) < 0.002
        a[pick] = (rng.integers(-1000, 1000, int(pick.sum())) * 1024).astype(a.dtype)
    return a


@pytest.mark.gpu
@pytest.mark.parametrize("content", ["smooth", "noise", "single"])
@pytest.mark.parametrize("mode", list(MODES_4D))
@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("n", [[4, 4, 4, 4], [15, 15, 4, 4], [17, 13, 5, 3], [28, 36, 4, 4], [6, 7, 41, 10]])
def test_4d_edges_gpu(n, tname, mode, content):
    from test_gpu_parity import check
    ztype = TYPES[tname]
    check(field_4d(n, ztype, content), n, ztype, MODES_4D[mode](ztype))
