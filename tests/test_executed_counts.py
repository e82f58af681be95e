"""The price of the coarsest inversion: at the size that is inverted, not at the
size that mhd_op_counts counts it by."""
import numpy as np
import pytest


@pytest.mark.parametrize("nc", [(4, 4, 3), (6, 4, 2)])
def test_dense_inversions_are_priced_at_the_condensed_size(nc):
    import cpu_baseline as cb
    from gridapmhd_amd import adjoint
    sp, _ = adjoint.inlet_duct(nc, 10.0, 5.0, 0.05)
    n1 = sp.nfree["u"] + sp.nfree["j"]
    inner = np.unique(sp.cell_dofs[:, 109:121])                # interior current dofs, one cell each
    kept = n1 - inner[(inner >= 0) & (inner < n1)].size
    counts = dict(setup_dense_dim3=2.0 * float(n1) ** 3, dense_entries=5.0)
    out = cb.executed_dense(counts, n1, sp.ncells)
    assert abs(out["setup_dense_dim3"] - 2.0 * float(kept) ** 3) <= 1e-12 * out["setup_dense_dim3"]
    assert out["dense_entries"] == 5.0 and counts["setup_dense_dim3"] == 2.0 * float(n1) ** 3
