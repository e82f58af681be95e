"""Calls of one context on several streams: a call whose header note allows it
to overlap others gives the bits it gives alone."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D2D, NON_BLOCKING = 3, 1


class Stream:
    """A non-blocking stream of the default priority."""

    def __enter__(self):
        from devmem import hip
        self.h = ctypes.c_void_p()
        assert hip().hipStreamCreateWithFlags(ctypes.byref(self.h), NON_BLOCKING) == 0
        return self.h.value

    def __exit__(self, *exc):
        from devmem import hip
        hip().hipStreamSynchronize(self.h)
        hip().hipStreamDestroy(self.h)


@pytest.mark.parametrize("kind", ["linear", "adjoint"])
def test_pending_residuals_beside_a_solve(kind):
    """Residuals that wait on a caller's stream, behind copies, while a linear or
    adjoint solve of the same context runs."""
    import gridapmhd_amd as g
    from devmem import DeviceArray, hip
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct((8, 8, 3), 20.0, 5.0, 0.05, convection="newton")
    rng = np.random.default_rng(12)
    x, rhs = 0.1 * rng.standard_normal(sp.ndofs), rng.standard_normal(sp.ndofs)
    ctx = g._lib.context_with_levels(sp, phys, levels=2)
    n, words = 24, 1 << 27
    try:
        solve = ctx.linear_solve if kind == "linear" else ctx.adjoint_solve
        o = ctx.default_opts(precision=1, ls_rtol=1e-10, max_krylov=400)
        alone = solve(x, rhs, o)[0]
        states = [DeviceArray.from_numpy(rng.standard_normal(sp.ndofs)) for _ in range(n)]
        out = [DeviceArray.from_numpy(np.full(sp.ndofs, np.nan)) for _ in range(n)]
        ref = []
        for s, r in zip(states, out):
            ctx.residual_d(s.ptr, r.ptr)
            ref.append(r.numpy())
            r.copy_from(np.full(sp.ndofs, np.nan))
        a, b = DeviceArray(words, np.float64), DeviceArray(words, np.float64)
        with Stream() as st:
            for s, r in zip(states, out):                     # about 0.5 ms of copies before every residual
                assert hip().hipMemcpyAsync(ctypes.c_void_p(b.ptr), ctypes.c_void_p(a.ptr),
                                            ctypes.c_size_t(a.nbytes), D2D, ctypes.c_void_p(st)) == 0
                ctx.residual_d(s.ptr, r.ptr, st)
            beside = solve(x, rhs, o)[0]
            got = [r.numpy() for r in out]
        print(f"[streams] {kind}: residuals that differ: {sum(not np.array_equal(p, q) for p, q in zip(got, ref))}, "
              f"solution differs: {not np.array_equal(alone, beside)}", flush=True)
        assert all(np.array_equal(p, q) for p, q in zip(got, ref))
        assert np.array_equal(alone, beside)
    finally:
        ctx.close()
