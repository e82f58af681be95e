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


def test_captured_product_after_another_assembly():
    """A product captured on the context's first stream (at a size where eager
    calls apply the form) is the product with the Jacobian of the replay's time."""
    import gridapmhd_amd as g
    from devmem import DeviceArray, hip
    sp, phys, rng = _problem((12, 12, 4))
    assert sp.ncells == 576
    v = rng.standard_normal(sp.ndofs)
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        assert ctx.nnz >= 5000000
        dx, dv, dy, dz = (DeviceArray.from_numpy(a) for a in (v, v, v, v))
        with Stream() as st:
            ctx.jacobian_d(dx.ptr, 0, st)
            ctx.spmv_d(dv.ptr, dz.ptr, st)
            graph = Graph(st, lambda: ctx.spmv_d(dv.ptr, dy.ptr, st))
            for k, conv in enumerate(("newton", "none", "picard", "newton")):
                p = dict(phys, gamma=phys["gamma"] * (k + 1), alpha=0.5 + k, zeta_u=float(k), convection=conv)
                x = 0.3 * rng.standard_normal(sp.ndofs)
                ctx.set_params(p)
                dx.copy_from(x)
                ctx.jacobian_d(dx.ptr, 0, st)
                ctx.spmv_d(dv.ptr, dz.ptr, st)                 # eager, the form applied
                graph.replay()
                y, z, ref = dy.numpy(), dz.numpy(), _product(g, sp, p, x, v)
                err = [np.linalg.norm(a - ref) / np.linalg.norm(ref) for a in (y, z)]
                print(f"[capture] product {conv}: replayed {err[0]:.2e}, eager {err[1]:.2e}", flush=True)
                assert max(err) < 1e-13
            graph.close()
    finally:
        ctx.close()


def test_product_after_a_replayed_assembly():
    """An assembly captured with some parameters and replayed after an eager one
    with others: the next product is with the replayed Jacobian."""
    import gridapmhd_amd as g
    from devmem import DeviceArray, hip
    sp, phys, rng = _problem((12, 12, 4))
    other = dict(phys, gamma=0.2 * phys["gamma"], alpha=3.0, convection="none")
    x, v = 0.3 * rng.standard_normal(sp.ndofs), rng.standard_normal(sp.ndofs)
    ref = {True: _product(g, sp, phys, x, v), False: _product(g, sp, other, x, v)}
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        dx, dv, dy = (DeviceArray.from_numpy(a) for a in (x, v, v))
        val = DeviceArray(ctx.nnz, np.float64)
        ctx.jacobian_d(dx.ptr, val.ptr)                        # the element buffer is there
        ctx.jacobian_d(dx.ptr, 0)
        ctx.spmv_d(dv.ptr, dy.ptr)
        assert hip().hipDeviceSynchronize() == 0
        with Stream() as st:
            graph = Graph(st, lambda: ctx.jacobian_d(dx.ptr, 0, st))
            ctx.set_params(other)
            for replayed in (False, True, True, False, True):
                if replayed:
                    graph.replay()
                else:
                    ctx.jacobian_d(dx.ptr, 0)
                ctx.spmv_d(dv.ptr, dy.ptr)
                y = dy.numpy()
                err = np.linalg.norm(y - ref[replayed]) / np.linalg.norm(ref[replayed])
                print(f"[capture] after {'a replayed' if replayed else 'an eager'} assembly: {err:.2e}", flush=True)
                assert err < 1e-13
            graph.close()
    finally:
        ctx.close()
