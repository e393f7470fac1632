import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an AMD MI355X (gfx950) GPU")


@pytest.fixture(scope="session")
def ctx():
    from zealot_amd import Context

    c = Context(0)
    yield c
    c.close()


def rel_amax(got, ref) -> float:
    """max |got - ref| / max |ref| (the cuTile self-test metric,
    src/biped/cutile_gemm.rs:733-739)."""
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    scale = max(float(np.max(np.abs(ref))) if ref.size else 0.0, 1e-30)
    return float(np.max(np.abs(got - ref))) / scale if ref.size else 0.0


def ulp_diff(a, b) -> int:
    """Max distance in units in the last place between two float32 arrays."""
    a = np.ascontiguousarray(a, np.float32).view(np.int32).astype(np.int64)
    b = np.ascontiguousarray(b, np.float32).view(np.int32).astype(np.int64)
    a = np.where(a < 0, -(a & 0x7FFFFFFF), a)
    b = np.where(b < 0, -(b & 0x7FFFFFFF), b)
    return int(np.max(np.abs(a - b))) if a.size else 0


def launches(ctx, fn, shapes=None):
    """Names of the kernels that fn launches, in order; (M, N, K, slices) of
    each GEMM launch (zeros of the others) appended to shapes."""
    import ctypes as C

    ctx.check(ctx.lib.zl_timing_begin(ctx.h, b"*"))
    fn()
    n = C.c_longlong()
    ctx.check(ctx.lib.zl_timing_end(ctx.h, None, C.byref(n), None))
    names = []
    for i in range(n.value):
        name, shape = C.c_char_p(), (C.c_int * 4)()
        ctx.check(ctx.lib.zl_timing_launch(ctx.h, i, C.byref(name), None, None, shape))
        names.append(name.value.decode())
        if shapes is not None:
            shapes.append(tuple(shape))
    return names
