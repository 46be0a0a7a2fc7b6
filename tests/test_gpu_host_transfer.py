"""Host transfers through pinned chunks: uploads and downloads on both sides of the one-chunk limit (256 KB) and
round the ring of chunks (16 MB), and the force's host matrices over several chunks."""
import numpy as np
import pytest

import grid_amd as gx
import npref as R

pytestmark = pytest.mark.gpu


def stored(a, prec):
    """What a field of this precision keeps of a, as complex128."""
    if prec == gx.F64:
        return a
    v = a.astype(np.complex64)
    if prec == gx.F32:
        return v.astype(np.complex128)
    r = v.reshape(-1, 12).view(np.float32).reshape(-1, 24)
    m = np.abs(r).max(1, keepdims=True)
    h = (r * (np.float32(1) / m)).astype(np.float16).astype(np.float32) * m
    return np.ascontiguousarray(h).view(np.complex64).reshape(a.shape).astype(np.complex128)


@pytest.mark.parametrize('prec', [gx.F64, gx.F32, gx.F16])
@pytest.mark.parametrize('dims,Ls,subset', [
    ((2, 2, 2, 2), 1, gx.FULL), ((2, 4, 2, 2), 3, gx.ODD), ((4, 6, 8, 7), 1, gx.FULL), ((8, 6, 4, 10), 7, gx.EVEN),
    ((8, 8, 8, 8), 2, gx.FULL), ((4, 4, 4, 4), 128, gx.ODD), ((16, 10, 12, 14), 5, gx.FULL)])
def test_round_trip(dims, Ls, subset, prec):
    ctx = gx.Context(0)
    a = gx.gaussian_fermion(dims, Ls, 41)
    if subset != gx.FULL:
        a = R.pick(a, dims, subset)
    f = gx.Field(ctx, dims, Ls, prec, subset)
    for shift in (0.0, 1.0):  # the second transfer reuses the chunks
        b = np.ascontiguousarray(a + shift)
        assert np.array_equal(f.upload(b).download(), stored(b, prec))
    f.close()
    ctx.close()


@pytest.mark.parametrize('dims,Ls', [((8, 8, 8, 16), 2), ((2, 2, 2, 4), 66), ((6, 4, 10, 4), 1)])
def test_force_chunks(dims, Ls):
    ctx = gx.Context(0)
    D = gx.FermionOp(ctx, gx.random_gauge(dims, 42, 0.4), dims, Ls, 'wilson', mass=0.1, phases=[1, 1, 1, -1])
    a, b = (gx.gaussian_fermion(dims, Ls, 43 + k) for k in (0, 1))
    A, B, leg = D.field().upload(a), D.field().upload(b), D.field()
    mat = D.DhopDeriv(A, B)
    ref = np.empty_like(mat)
    for mu in range(4):
        D.DhopDir(B, leg, mu, 1)
        ref[:, :, :, :, mu] = np.einsum('tzyxsia,tzyxsib->tzyxab', leg.download(), a.conj())
    # sums of 4 Ls products of terms of order one
    assert np.abs(mat - ref).max() < 1e-14 * 4 * Ls * np.abs(ref).max()
    par = np.indices(dims[::-1]).sum(0) % 2
    for which, ca in (('EO', 0), ('OE', 1)):
        ha, hb = (D.field(gx.F64, c) for c in (ca, 1 - ca))
        gx.pick_checkerboard(ca, ha, A)
        gx.pick_checkerboard(1 - ca, hb, B)
        half = D.DhopDeriv(ha, hb, 0, which)
        assert np.array_equal(half[par == ca], mat[par == ca]) and not half[par != ca].any()
    D.close()
    ctx.close()
