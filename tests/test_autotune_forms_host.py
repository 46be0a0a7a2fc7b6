"""CPU checks of the tuner's choice of launch form, with both timers injected: the hop's fastest form stays only where the
CG, whose reductions not every form folds in, does not lose by it; and small lattices keep the knobs that their
default hop ignores."""
import os
import re

import pytest

import grid_amd as gx
from grid_amd import autotune as at


class FakeField:
    def upload(self, a):
        return self

    def close(self):
        pass


class FakeOp:
    kind = 'wilson'

    def __init__(self, dims, Ls):
        self.dims, self.Ls = dims, Ls

    def field(self, prec, subset):
        return FakeField()


def tuned(dims, Ls, prec, hop, cg):
    """tune() with hop(knobs) and cg(knobs) as the times; knobs by name."""
    saved = {(k, p): gx.tune_get(k, p) for k in at.KNOB_NAMES for p in at.PRECS}

    def now():
        return {n: gx.tune_get(k, prec) for k, n in at.KNOB_NAMES.items()}

    t = at.Autotuner(ctx=None, cache_path=None, device='gfx950')
    t._time_dhop = lambda *a: hop(now())
    t._time_cg = lambda *a: cg(now())
    try:
        vals = t.tune(FakeOp(dims, Ls), prec, rounds=1)
        return {at.KNOB_NAMES[k]: v for k, v in vals.items()}
    finally:
        for (k, p), v in saved.items():
            gx.tune_set(k, v, p)


BIG, SMALL = (8, 8, 8, 24), (4, 4, 4, 4)   # 98304 and 2048 entries per checkerboard with Ls = 16


@pytest.mark.parametrize('prec', at.PRECS)
@pytest.mark.parametrize('form', [{'dhop_shape': 4, 'dhop_persist': 1}, {'dhop_tile': 1}])
def test_form_without_epilogues_gives_way(prec, form):
    is_form = lambda k: all(k[n] == v for n, v in form.items())
    got = tuned(BIG, 16, prec, lambda k: 0.9 if is_form(k) else 1.0, lambda k: 1.3 if is_form(k) else 1.0)
    assert not is_form(got)
    got = tuned(BIG, 16, prec, lambda k: 0.9 if is_form(k) else 1.0, lambda k: 0.9 if is_form(k) else 1.0)
    assert is_form(got)


# (FP32 and FP16 then also take the other prefetch setting for any gain in the CG, so 1% moves them)
@pytest.mark.parametrize('prec,loss,keep', [(gx.F64, 1.05, False), (gx.F32, 1.05, False), (gx.F16, 1.05, False), (gx.F64, 1.01, True)])
def test_wave_shape_against_the_folded_cg(prec, loss, keep):
    shaped = lambda k: k['dhop_shape'] == 4 and not k['dhop_persist']
    got = tuned(BIG, 16, prec, lambda k: 0.96 if shaped(k) else 1.0, lambda k: loss if shaped(k) else 1.0)
    assert shaped(got) == keep


@pytest.mark.parametrize('prec', at.PRECS)
def test_small_lattices_keep_ignored_knobs(prec):
    # the same kernel whatever these knobs say, with timing noise that favours others
    noise = lambda k: 1.0 + 0.1 * k['dhop_map'] + 0.1 * k['dhop_pf'] + 0.1 * k['dhop_nt']
    got = tuned(SMALL, 16, prec, lambda k: 2.0 if k['dhop_shape'] or k['dhop_tile'] else noise(k), lambda k: 1.0)
    assert (got['dhop_map'], got['dhop_pf'], got['dhop_nt'], got['dhop_order'], got['dhop_shape']) == (4, 1, 1, 0, 0)


def test_leg_per_wave_range():
    ask = at.leg_per_wave
    assert all(ask((8, 8, 8, 8), 16, p) for p in at.PRECS)            # 512 workgroups
    assert [ask((8, 8, 8, 9), 16, p) for p in at.PRECS] == [False, False, True]
    assert [ask((8, 8, 8, 10), 12, p) for p in at.PRECS] == [False, True, True]   # 512 of 60 lanes
    assert all(ask((16, 16, 16, 20), 1, p) for p in at.PRECS) and not any(ask((16, 16, 16, 22), 1, p) for p in at.PRECS)
    assert not any(ask((2, 2, 2, 2), 128, p) for p in at.PRECS)


def test_extent_without_tiles():
    got = tuned(SMALL, 33, gx.F64, lambda k: 1.0, lambda k: 1.0)
    assert got['dhop_shape'] == 0 and got['dhop_tile'] == 0


def test_split_range_is_the_librarys():
    with open(os.path.join(os.path.dirname(at.__file__), 'csrc', 'gx_internal.h')) as f:
        assert int(re.search(r'kSplitMax = (\d+);', f.read()).group(1)) == at.SPLIT_ENTRIES
    assert all(gx.tune_get(k, p) == v for k, v in at.HOP_DEFAULTS for p in at.PRECS)


def test_hop_only():
    """The hop's own winner stays where the program does not solve, whatever the CG takes."""
    saved = {(k, p): gx.tune_get(k, p) for k in at.KNOB_NAMES for p in at.PRECS}
    t = at.Autotuner(ctx=None, cache_path=None, device='gfx950')
    fast = lambda: gx.tune_get(gx.TUNE_DHOP_SHAPE) == 4 and gx.tune_get(gx.TUNE_DHOP_PERSIST) == 1
    t._time_dhop = lambda *a: 0.9 if fast() else 1.0
    t._time_cg = lambda *a: 1.3 if fast() else 1.0
    try:
        D = FakeOp(BIG, 16)
        assert t.tune(D, gx.F64, rounds=1, hop_only=True)[gx.TUNE_DHOP_PERSIST] == 1
        assert t.tune(D, gx.F64, rounds=1)[gx.TUNE_DHOP_PERSIST] == 0  # and is not kept for solves
    finally:
        for (k, p), v in saved.items():
            gx.tune_set(k, v, p)


def test_cached_workload_sets_its_precision_only():
    saved = {(k, p): gx.tune_get(k, p) for k in at.KNOB_NAMES for p in at.PRECS}
    t = at.Autotuner(ctx=None, cache_path=None, device='gfx950')
    t.cache[at.workload_key('gfx950', 'wilson', BIG, 16, gx.F32)] = {'knobs': {'dhop_map': 2}}
    try:
        assert t.tune(FakeOp(BIG, 16), gx.F32) == {gx.TUNE_DHOP_MAP: 2}
        assert [gx.tune_get(gx.TUNE_DHOP_MAP, p) for p in (gx.F64, gx.F32, gx.F16)] == [4, 2, 4]
    finally:
        for (k, p), v in saved.items():
            gx.tune_set(k, v, p)
