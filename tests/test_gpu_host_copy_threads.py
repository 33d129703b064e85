"""What a read-back of fields costs the host (csrc/host_copy.hip).  The ring and its
threads are for ordinary memory: a copy into memory that HIP knows (pinned by the
caller) goes there directly, and while the stream still has work none of the threads
runs.  Both show in the processor time of the read over its own duration: one waiting
thread uses at most the duration, and the runtime's own thread as much again; eight
threads use up to eight times it.  The bound of 3 lies between.
"""
import ctypes as C
import resource
import time

import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import F_Q, Block, lib

pytestmark = pytest.mark.gpu


def _cpu():
    r = resource.getrusage(resource.RUSAGE_SELF)
    return r.ru_utime + r.ru_stime


def _threads_busy(f):
    """processor time of f() per its duration"""
    c0, t0 = _cpu(), time.perf_counter()
    f()
    t1, c1 = time.perf_counter(), _cpu()
    return (c1 - c0) / (t1 - t0)


def _block(n):
    case = cases.smooth_box(n, n, n, viscous=0)
    b = Block(case.params)
    b.calc_metrics(case.x, case.y, case.z, case.period)
    b.set_conservative(cases.q_ref_aos(case))
    b.set_bc_calc_primitive(0)
    return b


def test_pinned_destination_takes_no_threads():
    hip = C.CDLL("libamdhip64.so")
    b = _block(128)
    nb = 5 * 8 * int(np.prod(b.shape))
    p = C.c_void_p()
    try:
        ref = b.get_field(F_Q, 5)
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t(nb), C.c_uint(0)) == 0
        dst = C.cast(p, C.POINTER(C.c_double))

        def read():
            for _ in range(40):
                assert lib().cbns_get_fields(b._h, F_Q, 5, dst) == 0

        read()
        busy = _threads_busy(read)
        print("threads busy", busy, flush=True)
        got = np.ctypeslib.as_array(dst, shape=(ref.size,)).reshape(ref.shape)
        assert np.array_equal(got, ref)
        # a destination inside the allocation
        assert lib().cbns_get_field(b._h, F_Q, C.cast(p.value + 4 * nb // 5,
                                                      C.POINTER(C.c_double))) == 0
        assert np.array_equal(got[4], ref[0])
        assert busy < 3.0
    finally:
        if p:
            hip.hipHostFree(p)
        b.free()


def test_queued_work_is_waited_for_by_one_thread():
    b = _block(64)
    try:
        b.get_field(F_Q, 5)  # the ring is there
        for _ in range(400):
            for s in (1, 2, 3):
                b.rk3_stage(0.0, s)
        out = []
        t0 = time.perf_counter()
        busy = _threads_busy(lambda: out.append(b.get_field(F_Q, 5)))
        print("read took", time.perf_counter() - t0, "threads busy", busy, flush=True)
        assert time.perf_counter() - t0 > 0.01  # the stages were still queued
        assert np.isfinite(out[0]).all()
        assert busy < 3.0
    finally:
        b.free()
