"""Row softmax over the edges of its kernels: rows that share a wave, a wave per
row, a work-group per row in registers (with unaligned rows and 1-3 columns
past the last quad), and rows beyond the registers."""
import ctypes as C

import numpy as np
import pytest

from camel_amd import _hip as H
from oracle import ffi as O
from tests import hipkit as K

pytestmark = pytest.mark.gpu

P = C.c_void_p
F = np.float32

# Short rows share a wave beyond 8192 + 32 cols rows (the last wave's rows are
# few); work-groups of 256 x 1, 2, 4, 8 and 512, 1024 x 8 quads; the three-pass
# kernel from 32769 columns on.
SHAPES = [(8193 + 32 * c, c) for c in (1, 2, 3, 4, 5, 8, 10, 16, 17, 32, 33, 63, 64, 65, 128, 132, 252, 256)]
SHAPES += [(8192, 10), (512, 513), (512, 1024), (513, 1023), (2048, 1025), (2049, 2048), (3, 2049),
           (5, 4095), (4, 4096), (7, 4097), (3, 8191), (2, 8192), (3, 8195), (2, 16384), (3, 16386),
           (2, 32767), (1, 32768), (2, 32769), (1, 70001)]


def run(x, offset=0):
    # `offset` floats into the buffers: rows that are only 4-byte aligned
    n = x.size
    flat = np.zeros(n + offset, F)
    flat[offset:] = x.ravel()
    dx, dy = K.dev(flat), K.empty((n + offset) * 4)
    H.call("camel_hip_softmax_rows", P(dx.ptr + 4 * offset), P(dy.ptr + 4 * offset), *x.shape)
    return K.host(dy, F, (n + offset,))[offset:].reshape(x.shape)


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_softmax_at_the_edges_of_its_kernels(rows, cols):
    # expf within 1 ulp, the sum rounded once from fp64, one rounded division:
    # 4 ulp of 2^-23, below the 1e-6 bar.  A row of special values each: -inf
    # is an exact 0, a NaN outside column 0 loses the max but enters the sum.
    print(f"softmax {rows}x{cols}", flush=True)
    rng = np.random.default_rng(rows * 7 + cols)
    x = rng.uniform(-20, 20, (rows, cols)).astype(F)
    x[-1, cols // 2:] = -np.inf if cols > 1 else x[-1, 0]
    ref = O.softmax_rows(x)
    for offset in (0, 1):
        got = run(x, offset)
        assert np.all(np.abs(got - ref) <= 1e-6 * np.abs(ref) + 1e-45), (rows, cols, offset)
    nan = x.copy()
    nan[0, 0] = np.nan
    nan[-1, -1] = np.nan
    got = run(nan)
    assert np.isnan(got[0]).all() and np.isnan(got[-1]).all()
    if rows > 2:
        assert np.array_equal(got[1:-1].view(np.uint32), run(x)[1:-1].view(np.uint32))
