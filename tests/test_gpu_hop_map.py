"""The blocked sweep (tile map 4), whose tiles cross block-slices, t wraps and y blocks, and the FP32 hop at two
workgroups per CU (fields beyond the Infinity Cache), against tiles in lattice order (map 0): every
entry takes the same arithmetic, so the same bits."""
import numpy as np
import pytest

import grid_amd as gx
import npref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('Ls,dims', [(16, (16, 16, 16, 6)), (7, (2, 2, 4, 2)), (12, (24, 24, 12, 32)), (5, (6, 10, 14, 12)),
                                     (3, (20, 36, 10, 14)), (24, (8, 20, 12, 10)), (4, (4, 34, 38, 6))])
def test_sweep_matches_lattice_order(Ls, dims):
    ctx = gx.Context(0)
    D = gx.FermionOp(ctx, gx.random_gauge(dims, 71, 0.3), dims, Ls, 'mobius', mass=0.1)
    f64 = D.field(gx.F64, gx.ODD).upload(R.pick(gx.gaussian_fermion(dims, Ls, 72), dims, gx.ODD))
    try:
        for prec in (gx.F64, gx.F32, gx.F16):
            src = D.field(prec, gx.ODD)
            gx.precision_change(src, f64)
            got = []
            for m in (4, 0):
                gx.tune_set(gx.TUNE_DHOP_MAP, m)
                e, o = D.field(prec, gx.EVEN), D.field(prec, gx.ODD)
                D.DhopEO(src, e, 1)
                D.MpcDagMpc(src, o)
                got.append([e.download(), o.download()])
            for a, b in zip(*got):
                assert np.array_equal(a, b) and np.isfinite(a).all() and np.abs(a).max() > 0
    finally:
        gx.tune_set(gx.TUNE_DHOP_MAP, 4)
        D.close()
        ctx.close()
