"""Host threads that share one context: its pinned chunks and block workspace serve one call at a time, so transfers, force
matrices and block products that run side by side each get their own data.  And block updates into fields of another context, which are complete on return."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import grid_amd as gx

pytestmark = pytest.mark.gpu


def each(n, f):
    with ThreadPoolExecutor(n) as ex:
        list(ex.map(f, range(n)))


@pytest.mark.parametrize('dims,Ls', [((4, 4, 4, 4), 2), ((8, 8, 12, 16), 8)])  # within the small chunk, round the ring of chunks
def test_transfers(dims, Ls):
    ctx = gx.Context(0)
    data = [gx.gaussian_fermion(dims, Ls, 100 + i) for i in range(4)]
    fields = [gx.Field(ctx, dims, Ls) for _ in range(4)]

    def work(i):
        for k in range(6):
            a = np.roll(data[i], k, axis=0)
            assert np.array_equal(fields[i].upload(a).download(), a), (i, k)

    each(4, work)
    ctx.close()


def test_block_products():
    dims, n = (8, 8, 8, 8), 6
    ctx = gx.Context(0)
    a = [gx.gaussian_fermion(dims, n, 110 + i) for i in range(8)]
    x = [gx.Field(ctx, dims, n).upload(v) for v in a]
    out = [gx.Field(ctx, dims, n) for _ in range(4)]
    col = [np.moveaxis(v, 4, 0).reshape(n, -1) for v in a]

    def work(i):
        rng = np.random.default_rng(i)
        u, v, cu, cv = x[i], x[4 + i], col[i], col[4 + i]
        m = cu.conj() @ cv.T
        for k in range(12):
            # sums of 49152 products of terms of order one, in another order
            assert np.abs(gx.slice_inner_product_matrix(u, v) - m).max() < 1e-13 * np.abs(cu.conj() @ cu.T).max(), (i, k)
            c = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
            gx.slice_madd_matrix(out[i], c, u, v, 0.5)
            got = np.moveaxis(out[i].download(), 4, 0).reshape(n, -1)
            assert np.abs(got - (cv + 0.5 * c.T @ cu)).max() < 1e-12, (i, k)

    each(4, work)
    ctx.close()


def test_updates_across_contexts():
    dims, n = (16, 16, 16, 16), 6
    one, two = gx.Context(0), gx.Context(0)
    a = gx.gaussian_fermion(dims, n, 120)
    x, y = gx.Field(one, dims, n).upload(a), gx.Field(two, dims, n).upload(a)
    r, z = gx.Field(two, dims, n), gx.Field(two, dims, n)
    c = np.eye(n)
    # slices as lists of fields of both contexts
    xs, rs = ([gx.Field(k, dims, 1).upload(np.ascontiguousarray(a[:, :, :, :, s:s + 1])) for s in range(n)] for k in (one, two))
    for k in range(1, 20):
        gx.slice_madd_matrix(r, k * c, x, y, 1.0)
        gx.axpby(z, 1.0, 0.0, r, r)  # on the other context's stream
        gx.madd_matrix(rs, c, xs, rs, 1.0)
        gx.axpby(rs[0], 0.5, 0.5, rs[0], rs[0])
    # small whole factors and halves: exact sums up to the rounding of one product each
    assert np.abs(z.download() - 20 * a).max() < 1e-13 * 20 * np.abs(a).max()
    for s in range(n):
        assert np.abs(rs[s].download()[..., 0, :, :] - 20 * a[..., s, :, :]).max() < 1e-13 * 20 * np.abs(a).max()
    one.close(), two.close()
