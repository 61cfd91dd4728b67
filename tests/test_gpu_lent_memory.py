"""Memory lent to a plan through the C ABI: a buffer that is replaced while a stream
of this thread is being captured, where the device cannot be waited for, is given
back after the capture and not during it; whatever was lent is back once the plan has
ended."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from tests import _cases as C

pytestmark = pytest.mark.gpu

THREAD_LOCAL = 1      # hipStreamCaptureModeThreadLocal


def test_a_replaced_buffer_is_waited_for(cuda):
    from quantem.gpu_amd.ssb.compute.hip import _abi
    lib = _abi.lib()
    pool = [cuda.empty(64 << 20, dtype=cuda.uint8, device="cuda") for _ in range(4)]
    lent, back = {}, []

    @_abi.AllocFn
    def alloc(nbytes, stream, ctx):
        if nbytes > pool[-1].numel():
            return None
        t = pool.pop()
        lent[t.data_ptr()] = t
        return t.data_ptr()

    @_abi.ReleaseFn
    def release(ptr, ctx):
        back.append(ptr)

    n, lam = 128, 0.0197
    plan = ctypes.c_void_p()
    stream = cuda.cuda.Stream()
    s = _abi.stream_handle(stream)
    _abi.call("ssb_plan_create_with", n, 32, 32, 16, lam, 21.4e-3, 1e-3, 1e-3, 0.5, 0.5, alloc, release, None, s,
              ctypes.byref(plan))
    case = C.make_engine_case(n, 9)
    rows, cols = (np.ascontiguousarray(v, np.int32) for v in (case.rows, case.cols))
    stacks = {k: cuda.from_numpy(np.ascontiguousarray(case.G[:k, :, :65])).cuda() for k in (5, 9)}
    cuda.cuda.synchronize()

    def load(num_bf):
        _abi.call("ssb_set_bf", plan, rows.ctypes.data_as(_abi._ip), cols.ctypes.data_as(_abi._ip), num_bf, 15.5, 15.5,
                  1.0, 0.0, s)

    load(5)
    _abi.call("ssb_import_g", plan, _abi.ptr(stacks[5]), 5, 65, s)
    stream.synchronize()
    load(9)
    lib.hipStreamBeginCapture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    lib.hipStreamEndCapture.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]
    lib.hipGraphDestroy.argtypes = [ctypes.c_void_p]
    graph = ctypes.c_void_p()
    assert lib.hipStreamBeginCapture(s, THREAD_LOCAL) == 0
    try:
        rc = lib.ssb_import_g(plan, _abi.ptr(stacks[9]), 9, 65, s)      # replaces the stack's buffer
        during = list(back)
    finally:
        lib.hipStreamEndCapture(s, ctypes.byref(graph))
        if graph.value:
            lib.hipGraphDestroy(graph)
    print("import under capture:", rc, "given back:", len(during))
    assert during == []
    cuda.cuda.synchronize()
    lib.ssb_plan_destroy(plan)
    assert sorted(back) == sorted(lent)
