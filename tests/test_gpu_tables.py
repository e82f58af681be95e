"""Dof and vertex tables that no mesher here makes but the interface takes."""
import dataclasses

import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def _u_dof_in_the_p_block(sp):
    """One velocity dof of the first cell numbered as a pressure dof of the last:
    outside of the [u,j] block, in a cell that does not hold it already."""
    cd = sp.cell_dofs.copy()
    k = [l for l in range(27) if cd[0, l] >= 0 and np.count_nonzero(cd == cd[0, l]) > 1][0]
    cd[0, k] = cd[-1, 82]
    return dataclasses.replace(sp, cell_dofs=cd)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["linear", "adjoint"])
@pytest.mark.parametrize("level", ["fine", "coarse"])
def test_velocity_dof_outside_of_its_block(level, kind, precision, orc_mod):
    """The residual that a solve reports is that of the oracle's system (the fine
    table altered: the preconditioner is a poor one, ten steps); on the coarsest
    level such a table leaves the solve converging."""
    import gridapmhd_amd as g
    from gridapmhd_amd import adjoint, fespaces, multigrid
    sp, phys = adjoint.inlet_duct((4, 4, 3), 10.0, 5.0, 0.05, convection="picard")
    rng = np.random.default_rng(5)
    bc = sp.bc_spec
    spc = fespaces.setup_fe_spaces(multigrid.coarsen_mesh(sp.mesh), bc["u_tags"], bc["j_tags"], bc["thin_walls"],
                                   style=sp.style)
    P, R = multigrid.prolongation(sp, spc)
    if level == "fine":
        sp = _u_dof_in_the_p_block(sp)
    else:
        spc = _u_dof_in_the_p_block(spc)
    x, rhs = 0.1 * rng.standard_normal(sp.ndofs), rng.standard_normal(sp.ndofs)
    A = orc_mod.Oracle(cases.problem_dict(sp, phys)).jacobian(x).tocsr()
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        ctx.attach_coarse(g._lib.context_from_spaces(spc, phys), P, R, 0, 0.175, "full")
        o = ctx.default_opts(precision=precision, ls_rtol=1e-10, max_krylov=400 if level == "coarse" else 10, restart=400)
        s, info, rc = (ctx.linear_solve if kind == "linear" else ctx.adjoint_solve)(x, rhs, o)
        r = (A if kind == "linear" else A.T.tocsr()) @ s - rhs
        if kind == "adjoint":  # measured with the j and phi rows over gamma / sigma
            fs = sp.field_slices()
            for f in ("j", "phi"):
                r[fs[f]] /= phys["gamma"] / phys["sigma"]
        print(f"[tables] u dof in the p block, {level}, {kind}, precision={precision}: rc={rc}, "
              f"{info.krylov_iters} iterations, residual {np.linalg.norm(r):.6e}, reported {info.residual:.6e}", flush=True)
        if level == "coarse":
            assert rc == 0 and np.linalg.norm(r) < 1e-9 * np.linalg.norm(rhs)
        else:
            assert abs(np.linalg.norm(r) - info.residual) < 1e-9 * np.linalg.norm(rhs)
    finally:
        ctx.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nz", [1, 2, 3])
def test_smoother_of_a_period_in_the_dof_table_only(nz, precision, orc_mod):
    """The two ends of a duct identified in the dof table but not in the vertex
    table: the patches of the end vertices hold dofs of cells that are not
    around them.  Against the full patches of the oracle's Jacobian."""
    import gridapmhd_amd as g
    from devmem import DeviceArray
    from test_gpu_condensation import _glued
    from test_gpu_solver import _vertex_patches
    sp = _glued((3, 2, nz))
    n = (nz + 1) * 12
    verts = np.unique(sp.mesh.cell_xyz().reshape(-1, 3).round(9), axis=0, return_inverse=True)[1]
    sp = dataclasses.replace(sp, cell_verts=verts.reshape(-1, 8).astype(sp.cell_verts.dtype))
    assert sp.cell_verts.max() + 1 == n
    phys = cases.cfd_physics(30.0, 10.0, zeta_u=1.0, zeta_j=1.0)
    rng = np.random.default_rng(9)
    x = 0.3 * rng.standard_normal(sp.ndofs)
    n1 = sp.nfree["u"] + sp.nfree["j"]
    A = orc_mod.Oracle(cases.problem_dict(sp, phys)).jacobian(x).tocsr()[:n1, :n1]
    r = rng.standard_normal(n1)
    ref = np.zeros(n1)
    patches = _vertex_patches(sp)
    for ids in patches:
        ref[ids] += np.linalg.solve(A[ids][:, ids].toarray(), r[ids])
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        ctx.jacobian(x)
        ctx.precond_setup(ctx.default_opts(precision=precision))
        dt = np.float64 if precision == 0 else np.float32
        rr, yy = DeviceArray.from_numpy(r, dt), DeviceArray.from_numpy(np.zeros(n1), dt)
        ctx.smoother_apply_d(rr.ptr, yy.ptr)
        err = np.linalg.norm(yy.numpy() - ref) / np.linalg.norm(ref)
        print(f"[tables] period of {nz} cells in the dof table only, precision={precision}: {len(patches)} patches, "
              f"rel err {err:.2e}", flush=True)
        # the bounds of the smoother test on full patches
        assert err < (1e-12 if precision == 0 else 1e-5)
    finally:
        ctx.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_dofs_in_no_cell_stay_zero(precision):
    """Three current dofs that no cell lists (empty rows): a solve leaves them zero
    and the others as they are without them."""
    import gridapmhd_amd as g
    from devmem import DeviceArray
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct((3, 3, 2), 10.0, 5.0, 0.05, convection="picard")
    n1, extra = sp.nfree["u"] + sp.nfree["j"], 3
    more = dataclasses.replace(sp, cell_dofs=np.where(sp.cell_dofs >= n1, sp.cell_dofs + extra, sp.cell_dofs).astype(np.int32),
                               nfree=dict(sp.nfree, j=sp.nfree["j"] + extra))
    rng = np.random.default_rng(5)
    x, rhs = 0.1 * rng.standard_normal(sp.ndofs), rng.standard_normal(sp.ndofs)
    pad = lambda v: np.concatenate([v[:n1], np.zeros(extra), v[n1:]])
    sol = []
    for s, a, b in ((sp, x, rhs), (more, pad(x), pad(rhs))):
        for _ in range(8):                                     # freed memory that holds other values than zero
            DeviceArray.from_numpy(np.full(1 << 20, 1e30))
        ctx = g._lib.context_from_spaces(s, phys)
        try:
            out, info, rc = ctx.linear_solve(a, b, ctx.default_opts(precision=precision, ls_rtol=1e-10, max_krylov=400,
                                                                    restart=400))
            assert rc == 0
            sol.append(out)
        finally:
            ctx.close()
    err = np.linalg.norm(np.delete(sol[1], range(n1, n1 + extra)) - sol[0]) / np.linalg.norm(sol[0])
    print(f"[tables] dofs in no cell, precision={precision}: {sol[1][n1:n1 + extra]}, others {err:.2e}", flush=True)
    assert np.all(sol[1][n1:n1 + extra] == 0.0) and err < 1e-7  # 1e-10 times the condition number's part


def test_a_refused_table_is_refused_again():
    """A solver that was refused half-way leaves nothing that a second call takes
    for a solver."""
    import gridapmhd_amd as g
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct((2, 2, 2), 10.0, 5.0, 0.05)
    cd = sp.cell_dofs.copy()
    cd[0, 82], cd[0, 83] = cd[0, 83], cd[0, 82]                # pressure dofs out of order
    ctx = g._lib.context_from_spaces(dataclasses.replace(sp, cell_dofs=cd), phys)
    try:
        x = np.zeros(sp.ndofs)
        o = ctx.default_opts()
        ctx.jacobian(x)
        for call in (lambda: ctx.precond_setup(o), lambda: ctx.precond_setup(o), lambda: ctx.newton_solve(x, o),
                     lambda: ctx.linear_solve(x, x, o)):
            with pytest.raises(g._lib.MhdError, match="p dofs of a cell must be consecutive"):
                call()
    finally:
        ctx.close()
