"""Batched ensembles (include/gmcore_ens.h) against per-member plain runs.

Bar: every member of the ensemble holds, after every step, exactly the bits
gmc_step gives the same member run on its own, for every launch shape the
tuner can pick; the tuner leaves the state where it found it.
"""
import numpy as np
import pytest

from helpers import STATE
from gmcore_amd import init_cond
from gmcore_amd.host import Ensemble, Setup, ShallowWater, make_config
from gmcore_amd.namelist import Namelist

pytestmark = pytest.mark.gpu

# (nlon, nlat, dt) of the members: uneven sizes, each with its own dt
MEMBERS = [(72, 37, 1800.0)] * 3 + [(144, 73, 900.0)] * 2 + [(180, 91, 600.0)]


def _member(nlon, nlat, dt, k, scheme="pc2"):
    st = Setup(Namelist(num_lon=nlon, num_lat=nlat, dt_dyn=dt, time_scheme=scheme))
    ic = init_cond.seeded_state(nlon, nlat, st.mesh.metrics, 8, 0, perturb=(0.01, 100 + k),
                                omega=st.nl.omega, radius=st.nl.radius)
    m = ShallowWater(st)
    m.set_state(*ic)
    m.prepare(1)
    return m


def _build(scheme="pc2"):
    return [_member(*spec, k, scheme) for k, spec in enumerate(MEMBERS)]


def _assert_same(ens_members, plain_members, what):
    for k, (a, b) in enumerate(zip(ens_members, plain_members)):
        assert a.level == b.level, (what, k)
        sa, sb = a.state(), b.state()
        for f in STATE:
            assert np.array_equal(sa[f], sb[f]), (what, k, f)


@pytest.mark.parametrize("scheme", ["pc2", "wrfrk3"])
def test_ensemble_equals_plain_runs(scheme):
    ens_m, plain = _build(scheme), _build(scheme)
    ens = Ensemble(ens_m)
    for n in range(3):
        ens.step(1)
        for m in plain:
            m.step(1)
        _assert_same(ens_m, plain, f"step {n}")
    ens.step(2)
    for m in plain:
        m.step(2)
    _assert_same(ens_m, plain, "step 5")
    # long runs replay graphs of 8 steps: from either parity, and the
    # members' own gmc_step runs in graphs of 8 steps as well
    for n in (10, 9):
        ens.step(n)
        for m in plain:
            for _ in range(n):
                m.step(1)
        _assert_same(ens_m, plain, f"{n} more steps")
    ens.close()


def test_every_shape_gives_the_same_bits():
    ref = _build()
    for m in ref:
        m.step(2)
    ncand = next(k for k in range(64) if not Ensemble.shape_name(k))
    assert ncand >= 6
    for shape in range(ncand):
        ms = _build()
        ens = Ensemble(ms)
        ens.set_shape(shape)
        ens.step(2)
        _assert_same(ms, ref, f"shape {shape} ({Ensemble.shape_name(shape)})")
        ens.close()


def test_autotune_keeps_state():
    ens_m, plain = _build(), _build()
    ens = Ensemble(ens_m)
    choice, times = ens.autotune(trial_steps=2)
    assert 0 <= choice < len(times) and np.all(times > 0)
    ens.step(3)
    for m in plain:
        m.step(3)
    _assert_same(ens_m, plain, f"after autotune (shape {choice})")
    ens.close()


# members whose rows all go through the filter kernels (narrow or low grids)
# beside members whose tiles take their short rows whole: the first sizes that
# do, odd and even zones, wide and hardly any filters, one and several segments
# of tile widths
ODD = [(62, 30, 1.0), (64, 23, 1.0), (64, 24, 1.0), (66, 25, 3.0), (108, 61, 1.0), (180, 91, 5.0), (502, 64, 1.0),
       (560, 65, 4.0), (722, 100, 0.2), (8, 5, 1.0)]


@pytest.mark.parametrize("shape", range(0, 9, 4))
def test_uneven_members_bitwise(shape):
    specs = [(nlon, nlat, 20000.0 * long / max(nlon, nlat)) for nlon, nlat, long in ODD]
    ens_m, plain = ([_member(*s, k) for k, s in enumerate(specs)] for _ in range(2))
    ens = Ensemble(ens_m)
    ens.set_shape(shape)
    for n in (1, 8):
        ens.step(n)
        for m in plain:
            m.step(n)
        _assert_same(ens_m, plain, f"{n} steps, shape {shape}")
    ens.close()


# the same beside a member of so many tiles that all members' short rows go
# through their tiles whole (512 tiles of 60 x 11 and more; the others above
# are some 300, every row in three kernels), and either side of that number
@pytest.mark.parametrize("more,shape", [((1440, 300, 1.0), 0), ((1440, 300, 1.0), 4), ((1440, 300, 1.0), 8),
                                        ((602, 198, 1.0), 0), ((602, 209, 1.0), 0)])
def test_uneven_members_whole_bitwise(more, shape):
    specs = [(nlon, nlat, 20000.0 * long / max(nlon, nlat)) for nlon, nlat, long in ODD + [more]]
    ens_m, plain = ([_member(*s, k) for k, s in enumerate(specs)] for _ in range(2))
    ens = Ensemble(ens_m)
    ens.set_shape(shape)
    ens.step(3)
    for m in plain:
        m.step(3)
    _assert_same(ens_m, plain, f"{more}, shape {shape}")
    ens.close()


def test_wide_filter_tables_bitwise():
    # tables of many more columns than any row has taps: what a launch keeps of
    # a row's weights is the row's taps
    def padded(nlon, nlat, dt, k):
        st = Setup(Namelist(num_lon=nlon, num_lat=nlat, dt_dyn=dt, time_scheme="pc2"))
        for f in (st.big, st.small):
            for w in ("wgt_lon", "wgt_lat"):
                a = getattr(f, w)
                wide = np.zeros((a.shape[0], 3000))
                wide[:, :a.shape[1]] = a
                setattr(f, w, wide)
            f.max_taps = 3000
        st.cfg = make_config(st.nl, st.big, st.small)
        ic = init_cond.seeded_state(nlon, nlat, st.mesh.metrics, 8, 0, perturb=(0.01, 100 + k),
                                    omega=st.nl.omega, radius=st.nl.radius)
        m = ShallowWater(st)
        m.set_state(*ic)
        m.prepare(1)
        return m

    specs = [(60, 31, 900.0), (180, 91, 600.0), (360, 181, 300.0), (720, 361, 150.0)]
    wide, alone, plain = ([make(*s, k) for k, s in enumerate(specs)] for make in (padded, padded, _member))
    ens = Ensemble(wide)
    ens.step(3)
    for m in alone + plain:
        m.step(3)
    _assert_same(wide, plain, "ensemble")
    _assert_same(alone, plain, "gmc_step")
    ens.close()


# members of one tile across (at most 60 columns) and several tiles high at
# every tile height, beside one two tiles across
NARROW = [(8, 30), (16, 40), (58, 30), (60, 31), (60, 12), (62, 30)]


@pytest.mark.parametrize("shape", range(9))
def test_narrow_members_bitwise(shape):
    specs = [(nlon, nlat, 20000.0 / max(nlon, nlat)) for nlon, nlat in NARROW]
    ens_m, plain = ([_member(*s, k) for k, s in enumerate(specs)] for _ in range(2))
    ens = Ensemble(ens_m)
    ens.set_shape(shape)
    ens.step(3)
    for m in plain:
        m.step(3)
    _assert_same(ens_m, plain, f"shape {shape}")
    ens.close()


@pytest.mark.parametrize("shape", [0, 1])
def test_tiles_of_every_launch_bitwise(shape):
    # more tiles than the filter launches have room for
    specs = [(180, 91, 600.0), (1440, 721, 60.0), (360, 181, 300.0)]
    ens_m, plain = ([_member(*s, k) for k, s in enumerate(specs)] for _ in range(2))
    ens = Ensemble(ens_m)
    ens.set_shape(shape)
    ens.step(2)
    for m in plain:
        m.step(2)
    _assert_same(ens_m, plain, f"shape {shape}")
    ens.close()
