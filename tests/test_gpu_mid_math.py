"""mid_rcp, mid_sqrt and mid_div equal the IEEE operation for every significand, at both ends of mid_range and
in its middle (both parities of the exponent, which a square root goes by), and mid_range holds where the
kernels rely on it and nowhere else."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libmid_math.so")


def apply(op, x):
    if not os.path.exists(LIB):
        import __graft_entry__
        __graft_entry__.build()
    L = ctypes.CDLL(LIB)
    L.mid_apply.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int]
    x = np.ascontiguousarray(x)
    out = np.empty_like(x)
    assert L.mid_apply(op, x.ctypes.data, out.ctypes.data, len(x)) == 0
    return out


OPS = {"rcp": (0, lambda x: np.float32(1.0) / x), "sqrt": (1, np.sqrt), "div5": (2, lambda x: x / np.float32(5.0)),
       "div6": (3, lambda x: x / np.float32(6.0))}


@pytest.mark.parametrize("exponent", [-80, -79, -24, -1, 0, 1, 23, 78, 79])
@pytest.mark.parametrize("name", list(OPS))
def test_every_significand(name, exponent):
    print("mid", name, exponent, flush=True)
    op, ieee = OPS[name]
    x = (np.arange(1 << 23, dtype=np.uint32) | np.uint32((exponent + 127) << 23)).view(np.float32)
    if exponent == 79:
        x = np.append(x, np.float32(2.0 ** 80))  # (the upper end)
    if name != "sqrt":
        x = np.concatenate([x, -x])
    got, want = apply(op, x), ieee(x)
    assert want.dtype == np.float32
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_range():
    low, high = np.float32(2.0 ** -80), np.float32(2.0 ** 80)
    inside = np.array([low, np.nextafter(low, high), 1.0, np.nextafter(high, low), high], dtype=np.float32)
    outside = np.array([0.0, 1e-45, np.finfo(np.float32).tiny, np.nextafter(low, np.float32(0)),
                        np.nextafter(high, np.float32(np.inf)), np.finfo(np.float32).max, np.inf, np.nan], dtype=np.float32)
    assert apply(4, np.concatenate([inside, -inside])).tolist() == [1.0] * 10
    assert apply(4, np.concatenate([outside, -outside])).tolist() == [0.0] * 16
