"""Assemblies and products of a context captured into a HIP graph: every replay,
with eager work between, gives what the eager calls give."""
import ctypes

import numpy as np
import pytest

from test_gpu_streams import Stream

pytestmark = pytest.mark.gpu


class Graph:
    """What `body` enqueues on `stream`, captured (no call of it may allocate)."""

    def __init__(self, stream, body):
        from devmem import hip
        self.h, self.stream = hip(), ctypes.c_void_p(stream)
        graph, self.exe = ctypes.c_void_p(), ctypes.c_void_p()
        assert self.h.hipStreamBeginCapture(self.stream, 0) == 0
        try:
            body()
        finally:
            rc = self.h.hipStreamEndCapture(self.stream, ctypes.byref(graph))
        assert rc == 0
        assert self.h.hipGraphInstantiate(ctypes.byref(self.exe), graph, None, None, ctypes.c_size_t(0)) == 0
        assert self.h.hipGraphDestroy(graph) == 0

    def replay(self):
        assert self.h.hipGraphLaunch(self.exe, self.stream) == 0
        assert self.h.hipStreamSynchronize(self.stream) == 0

    def close(self):
        assert self.h.hipGraphExecDestroy(self.exe) == 0


def _problem(nc, convection="newton", seed=3):
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct(nc, 20.0, 5.0, 0.05, convection=convection, jitter=0.15)
    return sp, phys, np.random.default_rng(seed)


def _product(g, sp, phys, x, v):
    """A(x) v of a context of its own, on its first stream."""
    from devmem import DeviceArray
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        dx, dv, dy = (DeviceArray.from_numpy(a) for a in (x, v, np.full(sp.ndofs, np.nan)))
        ctx.jacobian_d(dx.ptr)
        ctx.spmv_d(dv.ptr, dy.ptr)
        return dy.numpy()
    finally:
        ctx.close()


@pytest.mark.parametrize("nc,convection", [((4, 3, 3), "newton"), ((3, 3, 2), "none"), ((12, 12, 4), "picard")])
def test_first_assembly_into_the_context_under_capture(nc, convection):
    """The element buffer is there (an assembly into the caller's values made it);
    the first assembly into the context needs no other memory."""
    import gridapmhd_amd as g
    from devmem import DeviceArray, hip
    sp, phys, rng = _problem(nc, convection)
    v = rng.standard_normal(sp.ndofs)
    states = [0.3 * rng.standard_normal(sp.ndofs) for _ in range(3)]
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        dx, dv, dy = (DeviceArray.from_numpy(a) for a in (states[0], v, np.zeros(sp.ndofs)))
        val = DeviceArray(ctx.nnz, np.float64)
        ctx.jacobian_d(dx.ptr, val.ptr)
        assert hip().hipDeviceSynchronize() == 0
        with Stream() as st:
            graph = Graph(st, lambda: ctx.jacobian_d(dx.ptr, 0, st))
            for x in states + states[:1]:
                dx.copy_from(x)
                graph.replay()
                ctx.spmv_d(dv.ptr, dy.ptr)
                y, ref = dy.numpy(), _product(g, sp, phys, x, v)
                err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
                print(f"[capture] assembly {nc} {convection}: {err:.2e}", flush=True)
                assert err < 1e-13
            graph.close()
    finally:
        ctx.close()
