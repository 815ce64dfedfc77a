"""The entry point that allocates nothing (vct_mlp_forward_noalloc) against
vct_mlp_forward, through the C ABI.

Inputs and outputs are device buffers the test allocates itself (hipMalloc
through ctypes); the entry point reads the rows where they are.  Two calls in a
row, the second with fewer rows, must each equal vct_mlp_forward's output bit
for bit (the second call must not see rows the first left behind), as must
calls whose output lies inside the features and calls in flight at the same
time; more rows than VCT_MLP_NOALLOC_MAX_ROWS are rejected.
"""
from __future__ import annotations

import ctypes as C
import sys

import numpy as np
import pytest

from voxel_cone_tracing_amd import _lib as L
from voxel_cone_tracing_amd.context import Context

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


class DeviceBuffer:
    """hipMalloc'd device memory (the caller's buffers)."""

    hip = None

    def __init__(self, nbytes):
        if DeviceBuffer.hip is None:
            h = C.CDLL("libamdhip64.so")
            h.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
            h.hipFree.argtypes = [C.c_void_p]
            h.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
            h.hipDeviceSynchronize.argtypes = []
            DeviceBuffer.hip = h
        self.p = C.c_void_p()
        assert self.hip.hipMalloc(C.byref(self.p), C.c_size_t(nbytes)) == 0
        self.nbytes = nbytes

    def put(self, a):
        a = np.ascontiguousarray(a)
        assert a.nbytes <= self.nbytes
        assert self.hip.hipMemcpy(self.p, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), 1) == 0  # H2D

    def get(self, a):
        assert self.hip.hipMemcpy(a.ctypes.data_as(C.c_void_p), self.p, C.c_size_t(a.nbytes), 2) == 0  # D2H
        return a

    def free(self):
        self.hip.hipFree(self.p)


def test_noalloc_forward_equals_forward(gpu_available):
    rng = np.random.default_rng(5)
    p = (rng.standard_normal(L.MLP_PARAMS) * 0.2).astype(np.float32)
    sizes = [5000, 1000]  # the second call smaller than the first
    with Context(16, 16) as ctx:
        ctx.mlp_set_params(p)
        ctx.sync()
        dx = DeviceBuffer(max(sizes) * 34 * 4)
        dy = DeviceBuffer(max(sizes) * 3 * 4)
        try:
            for n in sizes:
                say(f"no-alloc forward, n={n}")
                x = rng.random((n, 34)).astype(np.float32) * 2 - 0.5
                want = ctx.mlp_forward(x)
                dx.put(x)
                dy.put(np.full((max(sizes), 3), np.nan, np.float32))
                L.check(ctx.lib.vct_mlp_forward_noalloc(ctx.h, dx.p, n, dy.p, None))
                ctx.sync()
                got = dy.get(np.zeros((max(sizes), 3), np.float32))
                assert np.array_equal(got[:n].view(np.uint32), want.view(np.uint32)), "differs from vct_mlp_forward"
                assert np.isnan(got[n:]).all(), "wrote past the n rows"
            rc = ctx.lib.vct_mlp_forward_noalloc(ctx.h, dx.p, L.MLP_NOALLOC_MAX_ROWS + 1, dy.p, None)
            assert rc == L.VCT_ERR_LIMIT
        finally:
            dx.free()
            dy.free()


@pytest.mark.parametrize("n,offset", [(1, 0), (33, 0), (5000, 0), (5000, -3), (5000, 33 * 5000), (5000, 34 * 5000 - 1),
                                      (L.MLP_NOALLOC_MAX_ROWS, 0), (L.MLP_NOALLOC_MAX_ROWS, 17 * 100_001)])
def test_noalloc_outputs_may_overlap_the_features(gpu_available, n, offset):
    """out inside features (offset in floats from their start), at either end
    and only 4-byte aligned: the outputs are vct_mlp_forward's, and what lies
    outside them keeps its bits."""
    say(f"no-alloc forward in place, n={n} offset={offset}")
    rng = np.random.default_rng(n + offset)
    p = (rng.standard_normal(L.MLP_PARAMS) * 0.2).astype(np.float32)
    x = (rng.random((n, 34)) * 2 - 0.5).astype(np.float32)
    pad = 4  # floats before the features and after the last output
    flat = np.concatenate([np.zeros(pad, np.float32), x.reshape(-1), np.zeros(3 * n + pad, np.float32)])
    with Context(16, 16) as ctx:
        ctx.mlp_set_params(p)
        ctx.sync()
        want = ctx.mlp_forward(x)
        d = DeviceBuffer(flat.nbytes)
        try:
            d.put(flat)
            L.check(ctx.lib.vct_mlp_forward_noalloc(ctx.h, d.p.value + 4 * pad, n, d.p.value + 4 * (pad + offset), None))
            ctx.sync()
            got = d.get(np.zeros_like(flat))
        finally:
            d.free()
    flat[pad + offset:pad + offset + 3 * n] = want.reshape(-1)
    assert np.array_equal(got.view(np.uint32), flat.view(np.uint32))


def test_noalloc_calls_on_two_streams(gpu_available):
    """Calls in flight at the same time on two streams, with inputs and row
    counts of their own, each give vct_mlp_forward's outputs."""
    say("no-alloc forward on two streams")
    rng = np.random.default_rng(6)
    p = (rng.standard_normal(L.MLP_PARAMS) * 0.2).astype(np.float32)
    xs = [(rng.random((n, 34)) * 2 - 0.5).astype(np.float32) for n in (200_003, 70_001)]
    with Context(16, 16) as ctx:
        ctx.mlp_set_params(p)
        ctx.sync()
        want = [ctx.mlp_forward(x) for x in xs]
        dx = [DeviceBuffer(x.nbytes) for x in xs]
        dy = [DeviceBuffer(w.nbytes) for w in want]
        hip = DeviceBuffer.hip
        streams = [C.c_void_p(), C.c_void_p()]
        try:
            for s in streams:
                assert hip.hipStreamCreateWithFlags(C.byref(s), C.c_uint(1)) == 0  # non-blocking, default priority
            for d, x in zip(dx, xs):
                d.put(x)
            for d, w in zip(dy, want):
                d.put(np.full_like(w, np.nan))
            for _ in range(8):
                for s, x, a, b in zip(streams, xs, dx, dy):
                    L.check(ctx.lib.vct_mlp_forward_noalloc(ctx.h, a.p, x.shape[0], b.p, s))
            for s in streams:
                assert hip.hipStreamSynchronize(s) == 0
            for d, w in zip(dy, want):
                assert np.array_equal(d.get(np.zeros_like(w)).view(np.uint32), w.view(np.uint32))
        finally:
            for s in streams:
                if s.value:
                    hip.hipStreamDestroy(s)
            for d in dx + dy:
                d.free()
