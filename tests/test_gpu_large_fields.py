"""The fifth-dimension operators on a half field of more than 2^32 stored complex numbers: their two bands act within
a site, so every slice is a sum of two slices of the input."""
import numpy as np
import pytest

import grid_amd as gx
import npref as R

pytestmark = pytest.mark.gpu


def test_bands_beyond_32_bits():
    dims, Ls, kw = (32, 32, 32, 176), 128, dict(mass=0.07, M5=1.8, b=1.5, c=0.5)
    lx, ly, lz, lt = dims
    half = lx * ly * lz * lt // 2
    assert 12 * half * Ls > 2 ** 32
    ctx = gx.Context(0)
    U = np.zeros((lt, lz, ly, lx, 4, 3, 3), dtype=np.complex128)
    U[..., range(3), range(3)] = 1
    D = gx.FermionOp(ctx, U, dims, Ls, 'mobius', **kw)
    del U
    rng = np.random.default_rng(81)
    a = np.empty((lt, lz, ly, lx // 2, 1, 4, 3), dtype=np.complex128)
    a.real, a.imag = (rng.random(a.shape, dtype=np.float32) - 0.5 for _ in range(2))
    parts = [np.roll(a, k, axis=0) for k in range(3)]
    psi, chi = D.field(gx.F32, gx.ODD), D.field(gx.F32, gx.ODD)
    one = [gx.Field(ctx, dims, 1, gx.F32, gx.ODD).upload(p) for p in parts]
    for s in range(Ls):
        gx.insert_slice(one[s % 3], psi, s)
    got = gx.Field(ctx, dims, 1, gx.F32, gx.ODD)
    Ap, Am = R.mooee_dense(Ls, kw['mass'], kw['M5'], kw['b'], kw['c'])
    for name, up, lo in (('Mooee', Ap, Am), ('MooeeDag', Ap.T, Am.T)):
        getattr(D, name)(psi, chi)
        for s in (0, 60, Ls - 1):
            gx.extract_slice(got, chi, s)
            g = got.download()
            print(name, s, flush=True)
            for spins, A in ((slice(0, 2), up), (slice(2, 4), lo)):
                ref = sum(A[s, t] * parts[t % 3][..., spins, :] for t in np.flatnonzero(A[s]))
                # two FP32 products and one sum of numbers below 4, everywhere
                assert np.abs(g[..., spins, :] - ref).max() < 2e-6, (name, s)
    for f in one + [got, psi, chi]:
        f.close()
    D.close()
    ctx.close()
