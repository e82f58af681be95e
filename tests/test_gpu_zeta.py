"""Negative weights of the div-div term, which make the interior current block of
a cell indefinite: nothing is eliminated then."""
import numpy as np
import pytest
import scipy.linalg as sla

import cases
from test_gpu_solver import _vertex_patches

pytestmark = pytest.mark.gpu


def _singular_zeta(orc_mod, sp, phys):
    """zeta_j at which the interior block of a cell is singular, the smallest in
    size (all cells are alike)."""
    i = np.sort(sp.cell_dofs[0, 109:121])
    M, D = (orc_mod.Oracle(cases.problem_dict(sp, dict(phys, zeta_j=z))).jacobian(np.zeros(sp.ndofs)).tocsr()[i][:, i].toarray()
            for z in (0.0, 1.0))
    return -1.0 / sla.eigh(D - M, M, eigvals_only=True).max()


@pytest.mark.parametrize("precision", [0, 1])
def test_smoother_where_the_interior_block_is_singular(precision, orc_mod):
    """Against the full patches of the oracle's Jacobian; then with a positive
    weight again on the same context (condensed), and back."""
    import gridapmhd_amd as g
    from devmem import DeviceArray
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct((3, 3, 2), 10.0, 5.0, 0.05, convection="picard")
    z = _singular_zeta(orc_mod, sp, phys)
    n1 = sp.nfree["u"] + sp.nfree["j"]
    rng = np.random.default_rng(4)
    x, r = 0.1 * rng.standard_normal(sp.ndofs), rng.standard_normal(n1)
    patches = _vertex_patches(sp)
    dt = np.float64 if precision == 0 else np.float32
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        for zeta in (z, 1.0, z):
            p = dict(phys, zeta_j=zeta)
            A = orc_mod.Oracle(cases.problem_dict(sp, p)).jacobian(x).tocsr()[:n1, :n1]
            ref, cond = np.zeros(n1), 0.0
            for ids in patches:
                M = A[ids][:, ids].toarray()
                cond = max(cond, np.linalg.cond(M))
                ref[ids] += np.linalg.solve(M, r[ids])
            ctx.set_params(p)
            ctx.jacobian(x)
            ctx.precond_setup(ctx.default_opts(precision=precision))
            rr, yy = DeviceArray.from_numpy(r, dt), DeviceArray.from_numpy(np.zeros(n1), dt)
            ctx.smoother_apply_d(rr.ptr, yy.ptr)
            err = np.linalg.norm(yy.numpy() - ref) / np.linalg.norm(ref)
            print(f"[zeta] {zeta:.6f}, precision={precision}: patch cond {cond:.1e}, rel err {err:.2e}", flush=True)
            # the vectors' rounding, and the patch solves' at their condition number
            assert err < (1e-14 if precision == 0 else 1e-6) + 33 * 1e-16 * cond
    finally:
        ctx.close()


def test_solves_with_changing_weights(orc_mod):
    """Linear and adjoint solves of one hierarchy with positive and negative
    weights in turn: the coarsest inverse is that of each."""
    import gridapmhd_amd as g
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct((4, 4, 2), 10.0, 5.0, 0.05, convection="picard")
    rng = np.random.default_rng(4)
    x, rhs = 0.1 * rng.standard_normal(sp.ndofs), rng.standard_normal(sp.ndofs)
    ctx = g._lib.context_with_levels(sp, phys, levels=2)
    try:
        o = ctx.default_opts(precision=0, ls_rtol=1e-10, max_krylov=400, restart=400)
        for zeta in (1.0, -1e-3, 1.0, -1e-3):
            p = dict(phys, zeta_j=zeta)
            A = orc_mod.Oracle(cases.problem_dict(sp, p)).jacobian(x).tocsr()
            ctx.set_params(p)
            for solve, M in ((ctx.linear_solve, A), (ctx.adjoint_solve, A.T.tocsr())):
                s, info, rc = solve(x, rhs, o)
                res = np.linalg.norm(M @ s - rhs) / np.linalg.norm(rhs)
                print(f"[zeta] solve {zeta}: {info.krylov_iters} iterations, residual {res:.2e}", flush=True)
                assert rc == 0 and res < 1e-9
    finally:
        ctx.close()
