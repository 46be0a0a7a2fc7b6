"""M and Mdag with the diagonal part in the hop's epilogue, and the banded fifth-dimension operators,
against the composition of the separate kernels (knob TUNE_FUSED off) in FP64."""
import numpy as np
import pytest

import grid_amd as gx
from conftest import max_site_rel_err

pytestmark = pytest.mark.gpu

# Both sides round a handful of sums of at most 20 terms: 1e-14 (FP64) and 1e-5 (FP32) leave two orders.
# FP16 storage keeps 2^-11 of a site's largest component; the worst site's norm may be a few times below
# the terms it is the sum of.
TOL = {gx.F64: 1e-14, gx.F32: 1e-5, gx.F16: 1e-2}


@pytest.mark.parametrize('prec', [gx.F64, gx.F32, gx.F16])
@pytest.mark.parametrize('kind,Ls,dims', [
    ('wilson', 1, (4, 4, 6, 4)), ('wilson', 5, (4, 6, 4, 4)), ('wilson', 24, (4, 4, 4, 4)),
    ('mobius', 2, (4, 4, 4, 6)), ('mobius', 3, (6, 4, 4, 4)), ('mobius', 11, (4, 4, 4, 4)),
    ('mobius', 16, (4, 4, 4, 4)), ('mobius', 24, (6, 4, 4, 4))])
def test_full_operator_fused(kind, Ls, dims, prec):
    ctx = gx.Context(0)
    U = gx.random_gauge(dims, 11, 0.4)
    D = gx.FermionOp(ctx, U, dims, Ls, kind, mass=0.07, phases=[1, 1, 1, -1])
    if kind == 'wilson' and Ls > 1:
        D.set_slice_masses([0.05 + 0.01 * s for s in range(Ls)])
    psi = gx.gaussian_fermion(dims, Ls, 12)
    fi = D.field(prec).upload(psi)
    rounded = D.field().upload(fi.download())  # the values both sides see
    out, ref = D.field(prec), D.field()
    for name in ('M', 'Mdag'):
        getattr(D, name)(fi, out)
        gx.tune_set(gx.TUNE_FUSED, 0)
        try:
            getattr(D, name)(rounded, ref)
        finally:
            gx.tune_set(gx.TUNE_FUSED, 1)
        assert max_site_rel_err(out.download(), ref.download()) < TOL[prec], name
    if kind == 'mobius':
        half = D.field(prec, gx.ODD)
        gx.pick_checkerboard(gx.ODD, half, fi)
        chi, again = D.field(prec, gx.ODD), D.field(prec, gx.ODD)
        inv = np.linalg.norm
        for there, back in (('Mooee', 'MooeeInv'), ('MooeeDag', 'MooeeInvDag')):  # banded, then dense
            getattr(D, there)(half, chi)
            getattr(D, back)(chi, again)
            a, b = again.download(), half.download()
            assert inv(a - b) < TOL[prec] * inv(b), there
    D.close()
    ctx.close()
