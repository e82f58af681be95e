"""The dense inverse of the coarsest level over sizes around its 96-wide block
columns, 192 x 96 workgroup tiles and 32-column panels: the set-up checks
A (A^-1 b) against b to 1e-6 and inverts again, by a pivoted LU, if that fails,
which the operation count shows.  A tile, remainder or pivot block gone wrong
leaves an error of order one.  The solve must satisfy the oracle's system."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc", [(2, 2, 1), (4, 2, 1), (4, 4, 1), (4, 4, 2), (6, 4, 3), (10, 6, 2), (8, 8, 3)])
def test_coarsest_inverse_needs_no_second_inversion(nc, orc_mod):
    import gridapmhd_amd as g
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct(nc, 10.0, 5.0, 0.05, convection="picard")
    x = 0.1 * np.random.default_rng(6).standard_normal(sp.ndofs)
    rhs = np.random.default_rng(7).standard_normal(sp.ndofs)
    A = orc_mod.Oracle(cases.problem_dict(sp, phys)).jacobian(x).tocsr()
    ctx = g._lib.context_with_levels(sp, phys, levels=2)
    try:
        o = ctx.default_opts(precision=0, ls_rtol=1e-10, max_krylov=400, restart=400)
        sol, info, rc = ctx.linear_solve(x, rhs, o)
        ctx.op_counts(reset=True)
        coarsest = sp._multigrid_cache[(0, 1)]["chain"][1]
        n1c = coarsest.nfree["u"] + coarsest.nfree["j"]
        res = np.linalg.norm(A @ sol - rhs) / np.linalg.norm(rhs)
        print(f"[coarse inverse] {nc}: n1c={n1c}, {info.krylov_iters} iterations, residual {res:.2e}", flush=True)
        assert rc == 0 and res < 1e-9
        o.max_newton = 1
        _, info, _ = ctx.newton_solve(x, o)  # counts its one inversion
        assert info.newton_iters == 1 and ctx.op_counts(reset=True)["setup_dense_dim3"] == float(n1c) ** 3
    finally:
        ctx.close()
