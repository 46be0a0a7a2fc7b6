"""The kernels of larger lattices on small ones: with the leg-per-wave hop off (TUNE_DHOP_SPLIT = 0), which otherwise takes
every lattice of up to 40960 entries, the tile maps, tile shapes and fused reductions run k_dhop and the general
tiles, against the same references.  The Ls = 1 cases hold its forms without staged links, with whole and partial
last tiles; two cases have more tiles than the folded iteration takes."""
import numpy as np
import pytest

import grid_amd as gx
import test_gpu_cg_fold as cg_fold
import test_gpu_full_fused as full_fused
import test_gpu_hop_map as hop_map
import test_gpu_mrhs_fused as mrhs_fused
import test_gpu_parity as parity

pytestmark = pytest.mark.gpu
system = mrhs_fused.system


@pytest.fixture(scope='module')
def ctx():
    c = gx.Context(0)
    yield c
    c.close()


@pytest.fixture(autouse=True)
def unsplit():
    gx.tune_set(gx.TUNE_DHOP_SPLIT, 0)
    yield
    gx.tune_set(gx.TUNE_DHOP_SPLIT, 1)


@pytest.mark.parametrize('kind,dims,Ls,prec', [('mobius', (8, 8, 8, 8), 16, gx.F64), ('wilson', (8, 4, 8, 8), 12, gx.F32),
                                               ('wilson', (8, 8, 4, 4), 1, gx.F64), ('mobius', (4, 6, 4, 8), 5, gx.F16)])
def test_tile_maps(ctx, kind, dims, Ls, prec):
    parity.test_tile_maps_bitwise(ctx, kind, dims, Ls, prec)


@pytest.mark.parametrize('Ls,dims', [(7, (2, 2, 4, 2)), (5, (6, 10, 14, 12)), (1, (6, 10, 14, 12))])
def test_sweep(Ls, dims):
    if Ls > 1:
        hop_map.test_sweep_matches_lattice_order(Ls, dims)
        return
    # one slice: map 4 stands for another map
    ctx = gx.Context(0)
    D = gx.FermionOp(ctx, gx.random_gauge(dims, 71, 0.3), dims, 1, 'wilson', mass=0.1)
    f, o = D.field().upload(gx.gaussian_fermion(dims, 1, 72)), D.field()
    got = []
    try:
        for m in (4, 0, 2):
            gx.tune_set(gx.TUNE_DHOP_MAP, m)
            D.M(f, o)
            got.append(o.download())
    finally:
        gx.tune_set(gx.TUNE_DHOP_MAP, 4)
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    D.close(), ctx.close()


@pytest.mark.parametrize('kind,Ls,dims', [('mobius', 8, (8, 4, 4, 8)), ('mobius', 16, (8, 4, 4, 8)), ('wilson', 12, (8, 4, 6, 8))])
@pytest.mark.parametrize('prec', [gx.F64, gx.F32, gx.F16])
def test_tile_shapes(ctx, kind, Ls, dims, prec):
    parity.test_tile_shapes_bitwise(ctx, kind, Ls, dims, prec)


@pytest.mark.parametrize('prec', [gx.F64, gx.F32, gx.F16])
@pytest.mark.parametrize('kind,Ls,dims', [('wilson', 1, (4, 4, 6, 4)), ('wilson', 5, (4, 6, 4, 4)), ('mobius', 2, (4, 4, 4, 6)),
                                          ('mobius', 11, (4, 4, 4, 4)), ('mobius', 24, (6, 4, 4, 4))])
def test_full_operator(kind, Ls, dims, prec):
    full_fused.test_full_operator_fused(kind, Ls, dims, prec)


@pytest.mark.parametrize('mixed', [1, 2])
def test_multi_rhs_reductions(ctx, system, mixed):
    mrhs_fused.test_fused_reductions_match_separate_passes(ctx, system, mixed)


@pytest.mark.parametrize('inner', [gx.F32, gx.F16])
def test_single_rhs_reductions(ctx, inner):
    mrhs_fused.test_single_rhs_fused_reductions(ctx, inner)


@pytest.mark.parametrize('kind,Ls,dims', [('wilson', 1, (4, 4, 6, 4)), ('wilson', 1, (6, 10, 14, 12)), ('wilson', 1, (32, 32, 32, 66)),
                                          ('wilson', 5, (16, 8, 12, 12)), ('mobius', 3, (4, 4, 4, 6)), ('mobius', 16, (8, 8, 12, 8)),
                                          ('mobius', 16, (20, 20, 20, 18)), ('mobius', 24, (8, 8, 8, 8))])
@pytest.mark.parametrize('graph', [0, 1])
def test_cg(kind, Ls, dims, graph):
    cg_fold.test_cg_fold(kind, Ls, dims, graph)


@pytest.mark.parametrize('maxit', [1, 8, 9])
def test_multishift_stopped(maxit):
    cg_fold.test_multishift_stopped(maxit)
