"""The one-leg-per-wave hop of small lattices gives the bits of the other tile shapes, with every epilogue,
for one checkerboard and for both in one launch."""
import numpy as np
import pytest

import grid_amd as gx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('prec', [gx.F64, gx.F32, gx.F16])
@pytest.mark.parametrize('kind,Ls,dims', [
    ('wilson', 1, (2, 2, 2, 2)), ('wilson', 1, (8, 6, 4, 8)), ('wilson', 5, (4, 6, 4, 4)), ('wilson', 33, (4, 4, 2, 4)),
    ('wilson', 64, (4, 4, 4, 2)), ('mobius', 2, (4, 4, 4, 6)), ('mobius', 7, (6, 4, 4, 4)), ('mobius', 16, (8, 4, 4, 6)),
    ('mobius', 24, (4, 4, 4, 4))])
def test_split_hop_bitwise(kind, Ls, dims, prec):
    ctx = gx.Context(0)
    U = gx.random_gauge(dims, 21, 0.4)
    D = gx.FermionOp(ctx, U, dims, Ls, kind, mass=0.07, phases=[1, 1, 1, -1])
    fi = D.field(prec).upload(gx.gaussian_fermion(dims, Ls, 22))
    odd, half, full = D.field(prec, gx.ODD), D.field(prec, gx.EVEN), D.field(prec)
    gx.pick_checkerboard(gx.ODD, odd, fi)
    calls = [('DhopEO', odd, half, (0,)), ('DhopEO', odd, half, (1,)), ('Dhop', fi, full, (0,)), ('Dhop', fi, full, (1,)),
             ('M', fi, full, ()), ('Mdag', fi, full, ()), ('Mpc', odd, half, ()), ('MpcDag', odd, half, ())]
    if Ls == 33:  # no whole-site tile of another shape holds an odd extent this large
        calls = []
        D.DhopEO(odd, half, 0)
        one = gx.FermionOp(ctx, U, dims, 1, kind, mass=0.07, phases=[1, 1, 1, -1])
        a, b = one.field(prec, gx.ODD), one.field(prec, gx.EVEN)
        x, y = odd.download(), half.download()
        for s in (0, 32):
            one.DhopEO(a.upload(x[:, :, :, :, s:s + 1]), b, 0)
            assert np.array_equal(b.download(), y[:, :, :, :, s:s + 1]), s
        one.close()
    for name, i, o, args in calls:
        got = []
        for split in (1, 0):
            gx.tune_set(gx.TUNE_DHOP_SPLIT, split)
            try:
                o.zero()
                getattr(D, name)(i, o, *args)
                got.append(o.download())
            finally:
                gx.tune_set(gx.TUNE_DHOP_SPLIT, 1)
        assert np.array_equal(got[0], got[1]), name
    D.close()
    ctx.close()
