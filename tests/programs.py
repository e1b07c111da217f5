"""Device programs put together step by step, for tests of the batch executors."""
import ctypes

import numpy as np

import qtorch_amd as qa
from qtorch_amd._native import _i32, hip

_vp = ctypes.c_void_p


class Program:
    """steps: (a, b, rank a, rank b, pairs, free) with operand ids and axes as
    qt_program_create takes them; leaf i lies at element offsets[i] of the pool."""

    def __init__(self, ctx, dim_log2, leaf_ranks, offsets, steps):
        desc, axes = [], []
        for a, b, ra, rb, pairs, free in steps:
            desc += [a, b, ra, rb, len(pairs), len(free)]
            axes += [x for x, _ in pairs] + [y for _, y in pairs]
            axes += [ax | qa.QT_FROM_A if from_a else ax for from_a, ax in free]
        refs = (ctypes.c_int64 * len(offsets))(*offsets)
        self.handle = _vp()
        ctx.check(hip.qt_program_create(ctx.handle, dim_log2, len(leaf_ranks), _i32(leaf_ranks), refs, len(steps),
                                        _i32(desc), _i32(axes), ctypes.byref(self.handle)), "qt_program_create")

    def scratch(self):
        elems = ctypes.c_int64()
        hip.qt_program_stats(self.handle, None, ctypes.byref(elems), None)
        return elems.value

    def __del__(self):
        hip.qt_program_destroy(self.handle)


class Batch:
    """One instance of each of `programs` (or of those named by `instances`) over `pool`."""

    def __init__(self, ctx, programs, precision, later=()):
        self.ctx, self.precision, self.n = ctx, precision, 0
        self.handle = _vp()
        handles = (_vp * max(len(programs), 1))(*[p.handle for p in programs])
        ctx.check(hip.qt_batch_create(ctx.handle, len(programs), handles, precision, ctypes.byref(self.handle)), "create")
        for p in later:
            ctx.check(hip.qt_batch_add_programs(self.handle, 1, (_vp * 1)(p.handle), (ctypes.c_int64 * 1)(0), None), "add")

    def set(self, pool, instances):
        v = np.ascontiguousarray(pool, dtype=np.complex128).view(np.float64)
        self.n = len(instances)
        self.ctx.check(hip.qt_batch_set_leaves(self.handle, v.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                                               len(pool)), "leaves")
        self.ctx.check(hip.qt_batch_set_instances(self.handle, self.n, _i32(instances), (ctypes.c_int64 * self.n)(), 0,
                                                  None, 0.0, 1.0), "instances")

    def set_outputs(self, tensors):
        self.ctx.check(hip.qt_batch_set_outputs(self.handle, len(tensors), (_vp * len(tensors))(*[t.handle for t in tensors])),
                       "outputs")

    def config(self, lanes, wgs, place=0):
        return hip.qt_batch_config_ex(self.handle, lanes, wgs, place)

    def shape(self):
        """(lanes, workgroups per CU, intermediates in device memory)"""
        lanes, wgs, place = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
        hip.qt_batch_info(self.handle, None, ctypes.byref(lanes), ctypes.byref(wgs), ctypes.byref(place), None)
        return lanes.value, wgs.value, bool(place.value & 1)

    def launch(self):
        self.ctx.check(hip.qt_batch_launch(self.handle), "launch")

    def results(self):
        v = np.zeros(2 * self.n)
        self.ctx.check(hip.qt_batch_results(self.handle, v.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), None), "results")
        return v.view(np.complex128)

    def run(self):
        self.launch()
        return self.results()

    def close(self):
        if self.handle:
            hip.qt_batch_destroy(self.handle)
            self.handle = None
