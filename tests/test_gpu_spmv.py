"""mhd_spmv_d from 5M nonzeros on, where the first stream that calls gets the form
applied cell by cell: the product is with the Jacobian as it was assembled,
whatever parameters and states the context has seen since."""
import numpy as np
import pytest

import cases
from test_gpu_streams import Stream

pytestmark = pytest.mark.gpu

_REF = {}


def _reference(orc_mod, nc, convection):
    """Spaces, physics, state, vector and the oracle's product (kept: 7M nonzeros)."""
    from gridapmhd_amd import adjoint
    if (nc, convection) not in _REF:
        sp, phys = adjoint.inlet_duct(nc, 20.0, 5.0, 0.05, convection=convection, jitter=0.15)
        rng = np.random.default_rng(8)
        x, v = 0.3 * rng.standard_normal(sp.ndofs), rng.standard_normal(sp.ndofs)
        A = orc_mod.Oracle(cases.problem_dict(sp, phys)).jacobian(x).tocsr()
        _REF[nc, convection] = sp, phys, x, v, A @ v
    return _REF[nc, convection]


@pytest.mark.parametrize("after", ["none", "picard", "newton"])
@pytest.mark.parametrize("nc,convection", [((12, 12, 4), "none"), ((12, 12, 4), "picard"), ((12, 12, 4), "newton"),
                                           ((13, 11, 5), "newton")])
def test_applied_product_is_the_assembled_jacobian(nc, convection, after, orc_mod):
    import gridapmhd_amd as g
    from devmem import DeviceArray, hip
    sp, phys, x, v, ref = _reference(orc_mod, nc, convection)
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        assert ctx.nnz >= 5000000
        dx, dv, dy = (DeviceArray.from_numpy(a) for a in (x, v, v))
        ctx.jacobian_d(dx.ptr)
        y = []
        with Stream() as other:
            for step in range(2):
                assert hip().hipDeviceSynchronize() == 0
                for stream in (0, other):
                    dy.copy_from(np.full(sp.ndofs, np.nan))
                    ctx.spmv_d(dv.ptr, dy.ptr, stream)
                    y.append(dy.numpy())
                ctx.residual(2.0 * x)                          # another state and other parameters in the context
                ctx.set_params(dict(phys, alpha=0.2, beta=3.0, gamma=3.0, sigma=0.5, zeta_u=7.0, zeta_j=0.3,
                                    B=np.array([0.3, -0.2, 0.8]), convection=after))
        err = [np.linalg.norm(a - ref) / np.linalg.norm(ref) for a in y]
        print(f"[spmv] {nc} {convection}, then {after}: applied {err[0]:.2e} {err[2]:.2e}, streamed {err[1]:.2e} "
              f"{err[3]:.2e}", flush=True)
        assert max(err) < 1e-13
        # the two routes (sums in another order) are taken, and neither changed
        assert not np.array_equal(y[0], y[1])
        assert np.array_equal(y[0], y[2]) and np.array_equal(y[1], y[3])
    finally:
        ctx.close()
