"""An upload replaces a field whole: what its padding entries held before (0 * inf = NaN after a non-finite factor, as a
diverged solve leaves it) does not reach later norms and products."""
import numpy as np
import pytest

import grid_amd as gx
import npref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('prec,tol', [(gx.F64, 1e-13), (gx.F32, 1e-6), (gx.F16, 2e-3)])
@pytest.mark.parametrize('dims,Ls,subset', [((2, 4, 2, 2), 3, gx.ODD), ((4, 2, 2, 3), 5, gx.FULL), ((6, 10, 6, 9), 7, gx.FULL),
                                            ((4, 4, 4, 2), 1, gx.EVEN)])
def test_upload_clears_padding(dims, Ls, subset, prec, tol):
    ctx = gx.Context(0)
    a = gx.gaussian_fermion(dims, Ls, 91)
    if subset != gx.FULL:
        a = R.pick(a, dims, subset)
    f, g = (gx.Field(ctx, dims, Ls, prec, subset).upload(a) for _ in range(2))
    gx.axpby(f, float('inf'), 1.0, f, g)
    f.upload(a)
    n2 = np.sum(np.abs(a) ** 2)
    assert abs(f.norm2() - n2) <= tol * n2
    assert abs(gx.inner_product(f, g) - n2) <= tol * n2
    f.close(), g.close(), ctx.close()
