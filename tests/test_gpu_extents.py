"""Which fifth-dimension extents an operator accepts does not depend on its lattice: Wilson operators take every Ls up to
64 (past 16 with an odd part above 7 through the leg-per-wave hop alone), Mobius ones refuse those in every call."""
import numpy as np
import pytest

import grid_amd as gx
import npref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('prec', [gx.F64, gx.F32, gx.F16])
@pytest.mark.parametrize('Ls', [22, 33, 57])
@pytest.mark.parametrize('dims', [(4, 4, 2, 4), (8, 8, 12, 6)])  # on both sides of 40960 entries
def test_wilson(dims, Ls, prec):
    ctx = gx.Context(0)
    U = gx.random_gauge(dims, 131, 0.3)
    D, one = (gx.FermionOp(ctx, U, dims, n, 'wilson', mass=0.2, phases=[1, 1, 1, -1]) for n in (Ls, 1))
    f, g = D.field(prec).upload(gx.gaussian_fermion(dims, Ls, 132)), D.field(prec)
    x, y = one.field(prec), one.field(prec)
    odd, out = D.field(prec, gx.ODD), D.field(prec, gx.ODD)
    gx.pick_checkerboard(gx.ODD, odd, f)
    a = f.download()
    try:
        for name, knobs in (('M', {}), ('Mdag', {gx.TUNE_DHOP_SPLIT: 0}), ('MpcDagMpc', {gx.TUNE_DHOP_SHAPE: 4})):
            for k, v in knobs.items():
                gx.tune_set(k, v)
            half = name == 'MpcDagMpc'
            getattr(D, name)(odd if half else f, out if half else g)
            gx.tune_set(gx.TUNE_DHOP_SPLIT, 1)
            gx.tune_set(gx.TUNE_DHOP_SHAPE, 0)
            got = (out if half else g).download()
            for s in (0, Ls - 1):
                x.upload(np.ascontiguousarray(a[:, :, :, :, s:s + 1]))
                if half:
                    xo, yo = one.field(prec, gx.ODD), one.field(prec, gx.ODD)
                    gx.pick_checkerboard(gx.ODD, xo, x)
                    one.MpcDagMpc(xo, yo)
                else:
                    yo = y
                    getattr(one, name)(x, y)
                assert np.array_equal(got[:, :, :, :, s:s + 1], yo.download()), (name, s)
    finally:
        gx.tune_set(gx.TUNE_DHOP_SPLIT, 1)
        gx.tune_set(gx.TUNE_DHOP_SHAPE, 0)
    if prec == gx.F64:
        r, sol = D.field(), D.field()
        st = D.schur_solve(f, sol, tol=1e-9)
        assert st['converged']
        D.M(sol, r)
        gx.axpby(r, 1.0, -1.0, r, f)
        assert r.norm2() < 1e-16 * f.norm2()
    D.close(), one.close(), ctx.close()


@pytest.mark.parametrize('Ls', [22, 33])
@pytest.mark.parametrize('dims', [(4, 4, 2, 4), (8, 8, 12, 8)])
def test_mobius_refuses(dims, Ls):
    ctx = gx.Context(0)
    D = gx.FermionOp(ctx, gx.random_gauge(dims, 133, 0.3), dims, Ls, 'mobius', mass=0.1)
    a = gx.gaussian_fermion(dims, Ls, 134)
    full, out = D.field().upload(a), D.field()
    odd, half = D.field(gx.F64, gx.ODD).upload(R.pick(a, dims, gx.ODD)), D.field(gx.F64, gx.EVEN)
    calls = [(n, full, out) for n in ('M', 'Mdag')] + [(n, odd, half) for n in (
        'Mpc', 'MpcDag', 'MpcDagMpc', 'Mooee', 'MooeeDag', 'MooeeInv', 'MooeeInvDag', 'Meooe', 'MeooeDag', 'M5D', 'Meooe5D')]
    for name, i, o in calls:
        with pytest.raises(RuntimeError, match='Ls'):
            getattr(D, name)(i, o)
    for name, i, o in (('Dhop', full, out), ('DhopEO', odd, half)):
        with pytest.raises(RuntimeError, match='Ls'):
            getattr(D, name)(i, o, 0)
    with pytest.raises(RuntimeError, match='Ls'):
        D.cg(odd, D.field(gx.F64, gx.ODD), tol=1e-8)
    with pytest.raises(RuntimeError, match='Ls'):
        D.schur_solve(full, out, tol=1e-8)
    D.close(), ctx.close()
