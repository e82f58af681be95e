"""The diagonal pivots of the patch inversions where a diagonal entry vanishes."""
import numpy as np
import pytest

import cases
from test_gpu_solver import _vertex_patches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rel", [0.0, 1e-12, 1e-6, -1e-3])
@pytest.mark.parametrize("nc", [(3, 3, 2), (2, 2, 1)])
def test_vanishing_diagonal_entry(nc, rel, orc_mod):
    """The convective derivative is scaled so that the first diagonal entry of one
    condensed patch matrix is `rel` times its value at rest.  Its row must not
    become the first pivot for being scaled by it: the smoother against the full
    patches, with the loss that the threshold allows (33 per pivot, 256 in a
    scaled row: under five digits of FP64's sixteen)."""
    import gridapmhd_amd as g
    from devmem import DeviceArray
    from gridapmhd_amd import adjoint
    sp, phys = adjoint.inlet_duct(nc, 10.0, 5.0, 0.05, convection="newton", jitter=0.1)
    n1 = sp.nfree["u"] + sp.nfree["j"]
    orc = orc_mod.Oracle(cases.problem_dict(sp, phys))
    rng = np.random.default_rng(17)
    step = rng.standard_normal(sp.ndofs)
    patches = _vertex_patches(sp)
    inner = np.zeros(n1, bool)
    inner[sp.cell_dofs[:, 109:121]] = True
    ids = max(patches, key=len)
    b, i = ids[~inner[ids]], ids[inner[ids]]

    def first(t):
        A = orc.jacobian(t * step).tocsr()
        return A[b[0], b[0]] - (A[b[:1]][:, i] @ np.linalg.solve(A[i][:, i].toarray(), A[i][:, b[:1]].toarray()))[0, 0]
    d0, d1 = first(0.0), first(1.0)
    x = (1.0 - rel) * d0 / (d0 - d1) * step
    A = orc.jacobian(x).tocsr()[:n1, :n1]
    r = rng.standard_normal(n1)
    ref, cond = np.zeros(n1), 0.0
    for p in patches:
        M = A[p][:, p].toarray()
        cond = max(cond, np.linalg.cond(M))
        ref[p] += np.linalg.solve(M, r[p])
    ctx = g._lib.context_from_spaces(sp, phys)
    try:
        ctx.jacobian(x)
        ctx.precond_setup(ctx.default_opts(precision=0))
        rr, yy = DeviceArray.from_numpy(r), DeviceArray.from_numpy(np.zeros(n1))
        ctx.smoother_apply_d(rr.ptr, yy.ptr)
        err = np.linalg.norm(yy.numpy() - ref) / np.linalg.norm(ref)
        print(f"[pivots] {nc} first entry {first((1.0 - rel) * d0 / (d0 - d1)) / d0:.1e} of its value at rest, "
              f"cond {cond:.1e}, {ctx.smoother_info(pivoted=True)[3]} partial pivoting: rel err {err:.2e}", flush=True)
        assert err < 33 * 256 * 1e-16 * cond
    finally:
        ctx.close()
