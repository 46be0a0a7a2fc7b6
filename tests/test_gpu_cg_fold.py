"""CG whose reductions fold into the hop, the last hop and the update (small lattices, and up to 4096 tile sums),
against CG on the separate passes (TUNE_FUSED off): the same solution in the same number of iterations."""
import numpy as np
import pytest

import grid_amd as gx
import npref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('graph', [0, 1])
@pytest.mark.parametrize('kind,Ls,dims', [('wilson', 1, (4, 4, 6, 4)), ('wilson', 1, (16, 16, 16, 20)), ('mobius', 3, (4, 4, 4, 6)),
                                          ('mobius', 7, (12, 8, 12, 12)), ('mobius', 16, (8, 8, 12, 8)), ('wilson', 5, (16, 8, 12, 12))])
def test_cg_fold(kind, Ls, dims, graph):
    ctx = gx.Context(0)
    D = gx.FermionOp(ctx, gx.random_gauge(dims, 51, 0.3), dims, Ls, kind, mass=0.2, phases=[1, 1, 1, -1])
    src = D.field(gx.F64, gx.ODD).upload(R.pick(gx.gaussian_fermion(dims, Ls, 52), dims, gx.ODD))
    shifts, got = [0.05, 0.3, 1.0], []
    try:
        gx.tune_set(gx.TUNE_CG_GRAPH, graph)
        for fused in (1, 0):
            gx.tune_set(gx.TUNE_FUSED, fused)
            x, s32, x32 = D.field(gx.F64, gx.ODD), D.field(gx.F32, gx.ODD), D.field(gx.F32, gx.ODD)
            a = D.cg(src, x, tol=1e-10)
            gx.precision_change(s32, src)
            b = D.cg(s32, x32, tol=1e-5)
            ms = [D.field(gx.F64, gx.ODD) for _ in shifts]
            c = D.cg_multishift(src, ms, shifts, [1e-10] * 3)
            assert a['converged'] and b['converged'] and all(k['converged'] for k in c)
            # maxit in the middle of a batch stops there
            y = D.field(gx.F64, gx.ODD)
            assert D.cg(src, y, tol=1e-30, maxit=5)['iterations'] == 5
            got.append(([a['iterations'], b['iterations']] + [k['iterations'] for k in c],
                        [x.download(), x32.download(), y.download()] + [f.download() for f in ms]))
    finally:
        gx.tune_set(gx.TUNE_FUSED, 1)
        gx.tune_set(gx.TUNE_CG_GRAPH, 1)
    for m, n in zip(got[0][0], got[1][0]):
        assert abs(m - n) <= 1, (got[0][0], got[1][0])
    # solutions to the tolerances asked for, times the condition of these systems (below 100)
    for u, v, tol in zip(got[0][1], got[1][1], (1e-8, 1e-3, 1e-10, 1e-8, 1e-8, 1e-8)):
        assert np.linalg.norm(u - v) < tol * np.linalg.norm(v)
    D.close()
    ctx.close()


@pytest.mark.parametrize('maxit', [1, 7, 8, 9, 19])
def test_multishift_stopped(maxit):
    """Stopped anywhere in a group of iterations, the unshifted system is at the iterate of CG (whose count
    includes the multishift's first one)."""
    dims, Ls = (8, 4, 6, 8), 4
    ctx = gx.Context(0)
    D = gx.FermionOp(ctx, gx.random_gauge(dims, 61, 0.3), dims, Ls, 'mobius', mass=0.1)
    src = D.field(gx.F64, gx.ODD).upload(R.pick(gx.gaussian_fermion(dims, Ls, 62), dims, gx.ODD))
    x, ms = D.field(gx.F64, gx.ODD), [D.field(gx.F64, gx.ODD) for _ in range(2)]
    D.cg(src, x, tol=1e-30, maxit=maxit + 1)
    st = D.cg_multishift(src, ms, [0.0, 1.0], [1e-30] * 2, maxit=maxit)
    assert not st[0]['converged'] and st[0]['iterations'] == maxit
    # 20 iterations of the same recurrences, rounded in another order
    assert np.linalg.norm(ms[0].download() - x.download()) < 1e-10 * np.linalg.norm(x.download())
    D.close()
    ctx.close()
