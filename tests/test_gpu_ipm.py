"""Inner-product matrices (slices of a field, lists of fields) for every number of columns that groups rows
differently on the matrix cores, against numpy, and several updates in a row through the kept workspace."""
import numpy as np
import pytest

import grid_amd as gx
import npref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('subset', [gx.FULL, gx.ODD])
@pytest.mark.parametrize('n,dims', [(1, (2, 2, 2, 2)), (2, (4, 2, 2, 6)), (3, (4, 6, 2, 2)), (5, (4, 4, 4, 4)), (6, (6, 4, 4, 4)),
                                    (8, (4, 4, 2, 2)), (9, (8, 4, 4, 6)), (12, (8, 8, 8, 8)), (16, (6, 4, 2, 4))])
def test_inner_product_matrices(n, dims, subset):
    ctx = gx.Context(0)
    a, b = (gx.gaussian_fermion(dims, n, 31 + k) for k in (0, 1))
    if subset != gx.FULL:
        a, b = R.pick(a, dims, subset), R.pick(b, dims, subset)
    x, y = (gx.Field(ctx, dims, n, gx.F64, subset).upload(v) for v in (a, b))
    ca, cb = (np.moveaxis(v, 4, 0).reshape(n, -1) for v in (a, b))
    # |sum of N products| rounds by at most eps sqrt(N) |x||y| in any order for such data; N <= 98304
    tol = 1e-13 * np.linalg.norm(ca[0]) * np.linalg.norm(cb[0])
    assert np.abs(gx.slice_inner_product_matrix(x, y) - ca.conj() @ cb.T).max() < tol
    assert np.abs(gx.slice_inner_product_matrix(x, x) - ca.conj() @ ca.T).max() < tol
    one = [[gx.Field(ctx, dims, 1, gx.F64, subset).upload(np.ascontiguousarray(v[:, :, :, :, s:s + 1])) for s in range(n)]
           for v in (a, b)]
    assert np.abs(gx.inner_product_matrix(*one) - ca.conj() @ cb.T).max() < tol
    # more updates in a row than the workspace has coefficient slots, none waited for
    r = gx.Field(ctx, dims, n, gx.F64, subset)
    gx.field_copy(r, x)
    rng = np.random.default_rng(5)
    ref = ca
    for k in range(20):
        m = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / (4 * n)
        gx.slice_madd_matrix(r, m, y, r, 1.0)
        ref = ref + m.T @ cb
    got = np.moveaxis(r.download(), 4, 0).reshape(n, -1)
    assert np.abs(got - ref).max() < 1e-12
    ctx.sync()
    for f in one[0] + one[1] + [x, y, r]:
        f.close()
    ctx.close()
