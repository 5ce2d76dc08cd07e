"""Uploads and downloads of arrays that are staged through pinned slots
(downloads from 16 MB, uploads from 32 MB) and of arrays just below: the
positions and B0 come back as they went up, bit for bit, also from several
threads at once, of which one at a time has the slots, and from and into
pinned memory, which is copied as it is."""
import threading

import numpy as np
import pytest

from conftest import small_braid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(require_gpu):
    import glemur_amd
    return glemur_amd


def round_trip(g, shape, seed, out):
    p = small_braid(*shape)
    r = np.random.default_rng(seed)
    n = 3 * (shape[0] + 2) * (shape[1] + 2) * (shape[2] + 2)
    B0, xb = r.random(n), r.random(n)
    with g.Context(p, g.PREC_F64) as c:
        for _ in range(2):
            c.upload(B0, xb, 0.0, 0.01)
            out.append(np.array_equal(c.download(g.FIELD_XB), xb) and np.array_equal(c.download(g.FIELD_B0), B0))
            B0, xb = xb, B0


# 16 MB and 32 MB lie at 699050 and 1398101 padded points; 33 MB is one chunk
# of 4 MB past eight, the largest wraps the slots twice
@pytest.mark.parametrize("shape", [(60, 62, 64), (86, 88, 86), (87, 87, 87), (110, 111, 107), (110, 112, 108),
                                   (118, 111, 109), (150, 140, 139)])
def test_round_trip(g, shape):
    out = []
    round_trip(g, shape, 1, out)
    assert out == [True, True]


def test_threads(g):
    out = []
    ts = [threading.Thread(target=round_trip, args=(g, (112, 112, 112), s, out)) for s in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert out == [True] * 6


def test_pinned_memory(g):
    import ctypes as C
    p = small_braid(112, 112, 112)
    n = 3 * 114 ** 3
    hip = g._lib                      # its HIP runtime is found through it
    ptr = [C.c_void_p(), C.c_void_p()]
    for q in ptr:
        assert hip.hipHostMalloc(C.byref(q), C.c_size_t(8 * n), C.c_uint(0)) == 0
    try:
        up, down = (np.ctypeslib.as_array(C.cast(q, C.POINTER(C.c_double)), (n,)) for q in ptr)
        up[:] = np.random.default_rng(5).random(n)
        down[:] = 0
        with g.Context(p, g.PREC_F64) as c:
            c.upload(up, up, 0.0, 0.01)
            assert g._lib.gm_download(c._h, g.FIELD_XB, C.cast(ptr[1], C.POINTER(C.c_double))) == 0
        assert np.array_equal(up, down)
    finally:
        for q in ptr:
            assert hip.hipHostFree(q) == 0
