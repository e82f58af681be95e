"""The vertex-star smoother with the cells' interior current dofs eliminated
(static condensation) against y = sum_P R_P^T A_P^-1 R_P r with the full patch
matrices of the oracle's Jacobian, where the elimination can go wrong:
a period of one cell (a cell lists dofs and vertices twice) and of two cells,
current Dirichlet faces (patches with few or no other dofs), an inlet / outlet
duct, a rotated unstructured mesh, and current dofs numbered at random
(interior dofs not consecutive: nothing is eliminated, 225-dof patches)."""
import dataclasses
import sys

import numpy as np
import pytest

import cases
from test_gpu_solver import _vertex_patches

pytestmark = pytest.mark.gpu


def _shuffled(sp, seed):
    """The same spaces with the free current dofs renumbered at random."""
    j = sp.field_slices()["j"]
    perm = np.arange(sp.ndofs)
    perm[j] = j.start + np.random.default_rng(seed).permutation(j.stop - j.start)
    cd = np.where(sp.cell_dofs >= 0, perm[np.maximum(sp.cell_dofs, 0)], sp.cell_dofs).astype(np.int32)
    return dataclasses.replace(sp, cell_dofs=cd)


def _glued(nc, **kw):
    """A duct with its two ends identified by hand: a period of nc[2] cells (the meshers start at three)."""
    mesh = g_meshers().cartesian_model((-1.0, 1.0, -1.0, 1.0, 0.0, 0.3), nc, (False, False, False))
    g_meshers().hunt_add_tags(mesh)
    sp = g_spaces().setup_fe_spaces(mesh, "walls", [], [dict(domain="walls", cw=0.05, tau=100.0, jw=0.0)],
                                    style="badia2024")
    cd, verts = sp.cell_dofs.copy(), sp.cell_verts.copy()
    per = nc[0] * nc[1]
    low, top = np.arange(per), np.arange(sp.ncells - per, sp.ncells)
    to = np.arange(sp.ndofs)                                   # top dof -> bottom dof
    lu = [[c * 27 + 9 * k + a for c in range(3) for a in range(9)] for k in (0, 2)]
    for lo, hi in ((lu[0], lu[1]), (range(85, 89), range(89, 93))):
        a, b = cd[low][:, list(lo)].ravel(), cd[top][:, list(hi)].ravel()
        free = b >= 0
        to[b[free]] = a[free]
    keep = np.unique(to)
    new = np.full(sp.ndofs, -1)
    new[keep] = np.arange(keep.size)
    nfree = {f: int(np.isin(np.arange(s.start, s.stop), keep).sum()) for f, s in sp.field_slices().items()}
    vto = np.arange(verts.max() + 1)
    vto[verts[top][:, 4:].ravel()] = verts[low][:, :4].ravel()
    return dataclasses.replace(sp, cell_dofs=np.where(cd >= 0, new[to[np.maximum(cd, 0)]], cd).astype(np.int32),
                               nfree=nfree, cell_verts=vto[verts])


def g_meshers():
    import gridapmhd_amd as g
    return g.meshers


def g_spaces():
    import gridapmhd_amd as g
    return g.fespaces


def _case(name):
    duct = lambda nc, **kw: cases.duct_thin_wall_case(nc, Ha=30.0, Re=10.0, cw=0.05, convection="newton",
                                                      style="badia2024", zeta_u=1.0, zeta_j=1.0, **kw)
    if name == "period_one_cell":
        return _glued((3, 2, 1)), cases.cfd_physics(30.0, 10.0, zeta_u=1.0, zeta_j=1.0)
    if name == "period_two_cells":
        return _glued((2, 3, 2)), cases.cfd_physics(30.0, 10.0, zeta_u=1.0, zeta_j=1.0)
    if name == "insulating":
        sp, phys = cases.hunt_case(3, Ha=30.0, nz=3, style="badia2024")
        return sp, dict(phys, zeta_u=1.0, zeta_j=1.0)
    if name == "inlet":
        from gridapmhd_amd import adjoint
        return adjoint.inlet_duct((3, 3, 2), 30.0, 10.0, 0.02, jitter=0.15)
    if name == "expansion":
        _, sp, phys = cases.expansion_case("expansion_710_thin_wall")
        return sp, dict(phys, zeta_u=1.0, zeta_j=1.0)
    sp, phys = duct((4, 3, 3))
    return _shuffled(sp, 3), phys


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", ["period_one_cell", "period_two_cells", "insulating", "inlet", "expansion",
                                  "not_consecutive"])
def test_condensed_smoother_matches_full_patches(name, precision, orc_mod):
    import gridapmhd_amd as g
    from devmem import DeviceArray
    sp, phys = _case(name)
    print(f"[condensation] {name} precision={precision} ndofs={sp.ndofs}", flush=True)
    rng = np.random.default_rng(9)
    x = 0.3 * rng.standard_normal(sp.ndofs)
    n1 = sp.nfree["u"] + sp.nfree["j"]
    A = orc_mod.Oracle(cases.problem_dict(sp, phys)).jacobian(x).tocsr()[:n1, :n1]
    patches = _vertex_patches(sp)
    r = rng.standard_normal(n1)
    y0 = rng.standard_normal(n1)
    y_ref = y0.copy()
    for ids in patches:
        y_ref[ids] += np.linalg.solve(A[ids][:, ids].toarray(), r[ids])
    for tau in (0.03, 1.0):           # diagonal pivots; partial pivoting of (nearly) every patch
        ctx = g._lib.context_from_spaces(sp, phys)
        try:
            ctx.set_pivot_threshold(tau)
            ctx.jacobian(x)
            ctx.precond_setup(ctx.default_opts(precision=precision))
            assert ctx.smoother_info() == (len(patches), max(p.size for p in patches), sum(p.size ** 2 for p in patches))
            dt = np.float64 if precision == 0 else np.float32
            rr, yy = DeviceArray.from_numpy(r, dt), DeviceArray.from_numpy(y0, dt)
            ctx.smoother_apply_d(rr.ptr, yy.ptr)
            y = yy.numpy().astype(np.float64)
        finally:
            ctx.close()
        err = np.linalg.norm(y - y_ref) / np.linalg.norm(y_ref)
        print(f"  tau={tau}: {len(patches)} patches, rel err {err:.2e}", flush=True)
        # the bounds of the smoother test on full patches
        assert err < (1e-12 if precision == 0 else 1e-5)
    sys.stdout.flush()
