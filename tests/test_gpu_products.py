"""The Jacobian products that the Krylov solves use (the form applied cell by
cell; with a skeleton term, the matrix) against the oracle's Jacobian: a
linear solve with A(x), or with its transpose, to a relative residual of 1e-11
must satisfy the oracle's system to the same residual.  Odd cell counts (the
last workgroup holds one cell), non-affine cells, every convection form, a
state with all fields, the [u,j] V-cycle's products in both precisions."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nc,convection,stab,levels", [((3, 3, 3), "newton", 0.0, 1), ((3, 2, 3), "picard", 0.0, 1),
                                                       ((5, 3, 1), "none", 0.0, 1), ((8, 8, 3), "newton", 0.0, 2),
                                                       ((3, 3, 3), "newton", 0.1, 1)])
def test_linear_solves_satisfy_the_oracle_system(nc, convection, stab, levels, precision, orc_mod):
    import gridapmhd_amd as g
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct(nc, 20.0, 5.0, 0.05, convection=convection, jitter=0.15 if levels == 1 else 0.0)
    phys = dict(phys, stab_mu=stab, f0=np.array([0.2, -0.1, 1.0]))
    rng = np.random.default_rng(4)
    x = 0.1 * rng.standard_normal(sp.ndofs)
    rhs = rng.standard_normal(sp.ndofs)
    A = orc_mod.Oracle(cases.problem_dict(sp, phys)).jacobian(x).tocsr()
    ctx = g._lib.context_with_levels(sp, phys, levels=levels)
    try:
        o = ctx.default_opts(precision=precision, ls_rtol=1e-11, max_krylov=600, restart=600, inner_iters=4)
        for name, solve, M in (("A", ctx.linear_solve, A), ("A^T", ctx.adjoint_solve, A.T.tocsr())):
            s, info, rc = solve(x, rhs, o)
            res = np.linalg.norm(M @ s - rhs) / np.linalg.norm(rhs)
            print(f"[products] {nc} {convection} stab={stab} precision={precision} {name}: {info.krylov_iters} "
                  f"iterations, residual {res:.2e}", flush=True)
            assert rc == 0
            # the adjoint solve measures its residual in rows scaled by up to gamma / sigma = Ha^2 / Re = 80
            assert res < 1e-9
    finally:
        ctx.close()


@pytest.mark.parametrize("nc,convection,stab", [((3, 3, 3), "newton", 0.0), ((5, 3, 1), "picard", 0.0),
                                                ((2, 2, 2), "none", 0.0), ((3, 2, 3), "newton", 0.1)])
def test_spmv_is_the_assembled_jacobian(nc, convection, stab, orc_mod):
    """mhd_spmv_d on the first stream that calls it (the form applied cell by
    cell) and on another (the matrix streamed): both are the Jacobian as it was
    assembled, whatever parameters and states the context has seen since."""
    import ctypes
    import gridapmhd_amd as g
    from devmem import DeviceArray, hip
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct(nc, 20.0, 5.0, 0.05, convection=convection, jitter=0.15)
    phys = dict(phys, stab_mu=stab)
    rng = np.random.default_rng(8)
    x, v = 0.3 * rng.standard_normal(sp.ndofs), rng.standard_normal(sp.ndofs)
    ref = orc_mod.Oracle(cases.problem_dict(sp, phys)).jacobian(x).tocsr() @ v
    other = ctypes.c_void_p()
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        assert hip().hipStreamCreate(ctypes.byref(other)) == 0
        dx, dv, dy = DeviceArray.from_numpy(x), DeviceArray.from_numpy(v), DeviceArray.from_numpy(np.zeros(sp.ndofs))
        ctx.jacobian_d(dx.ptr)
        ctx.residual(2.0 * x)                                      # another state in the context
        ctx.set_params(dict(phys, gamma=3.0, alpha=0.2, convection="newton"))
        hip().hipDeviceSynchronize()
        for stream in (0, other.value, 0):
            dy.copy_from(np.full(sp.ndofs, np.nan))
            ctx.spmv_d(dv.ptr, dy.ptr, stream)
            err = np.linalg.norm(dy.numpy() - ref) / np.linalg.norm(ref)
            print(f"[spmv] {nc} {convection} stab={stab} stream={'own' if not stream else 'other'}: {err:.2e}", flush=True)
            assert err < 1e-13
    finally:
        ctx.close()
        hip().hipStreamDestroy(other)


@pytest.mark.parametrize("nc", [(12, 10, 4), (12, 12, 4), (13, 11, 5)])
def test_spmv_routes_agree_around_their_line(nc):
    """Below 5M nonzeros both streams stream the matrix (the same bits), from
    there on the first stream applies the form: sums of at most 700 products in
    another order, on rows of entries of one size."""
    import ctypes
    import gridapmhd_amd as g
    from devmem import DeviceArray, hip
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct(nc, 20.0, 5.0, 0.05, convection="newton", jitter=0.15)
    rng = np.random.default_rng(9)
    x, v = 0.3 * rng.standard_normal(sp.ndofs), rng.standard_normal(sp.ndofs)
    other = ctypes.c_void_p()
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        assert hip().hipStreamCreate(ctypes.byref(other)) == 0
        dx, dv, dy = DeviceArray.from_numpy(x), DeviceArray.from_numpy(v), DeviceArray.from_numpy(np.zeros(sp.ndofs))
        ctx.jacobian_d(dx.ptr)
        hip().hipDeviceSynchronize()
        y = {}
        for stream in (0, other.value):
            dy.copy_from(np.full(sp.ndofs, np.nan))
            ctx.spmv_d(dv.ptr, dy.ptr, stream)
            y[stream] = dy.numpy().copy()
        err = np.linalg.norm(y[0] - y[other.value]) / np.linalg.norm(y[0])
        print(f"[spmv routes] {nc}: nnz {ctx.nnz}, {err:.2e}", flush=True)
        assert (err == 0.0) == (ctx.nnz < 5000000) and err < 1e-13
    finally:
        ctx.close()
        hip().hipStreamDestroy(other)
