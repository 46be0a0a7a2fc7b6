"""Where the leg-per-wave hop ends: lattices past one round of its workgroups, of whose solves some hops run one leg per
wave and others in 4-wave tiles, and the times of both forms there."""
import pytest

import grid_amd as gx
import test_gpu_cg_fold as cg_fold

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('kind,Ls,dims', [('wilson', 12, (8, 8, 8, 12)), ('mobius', 10, (8, 8, 8, 16)), ('wilson', 4, (8, 8, 16, 18)),
                                          ('mobius', 16, (8, 8, 8, 10)), ('mobius', 24, (4, 10, 8, 10))])
def test_cg(kind, Ls, dims):
    cg_fold.test_cg_fold(kind, Ls, dims, 1)


@pytest.mark.parametrize('Ls,dims', [(12, (8, 8, 8, 12)), (10, (8, 8, 8, 16))])
def test_not_slower_than_tiles(Ls, dims):
    """FP64, 615 and 683 workgroups: one leg per wave took 1.4 times the tiles' time; the default takes theirs."""
    ctx = gx.Context(0)
    D = gx.FermionOp(ctx, gx.random_gauge(dims, 1, 0.3), dims, Ls, 'wilson', mass=0.1)
    f, o = D.field(gx.F64, gx.ODD), D.field(gx.F64, gx.EVEN)
    best = {0: 1e9, 1: 1e9}
    try:
        for _ in range(8):
            for split in best:
                gx.tune_set(gx.TUNE_DHOP_SPLIT, split)
                D.DhopEO(f, o, 0)
                ctx.sync()
                ctx.record(0)
                for _ in range(50):
                    D.DhopEO(f, o, 0)
                ctx.record(1)
                ctx.sync()
                best[split] = min(best[split], ctx.elapsed_ms(0, 1))
    finally:
        gx.tune_set(gx.TUNE_DHOP_SPLIT, 1)
    assert best[1] < 1.2 * best[0], best
    D.close(), ctx.close()
