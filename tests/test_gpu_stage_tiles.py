"""The fused stage at the edges of its tiles and bands.

Bar: 1e-12 relative against the oracle (the per-step bar of the SW fields),
and bit equality between the forms of a stage, whose expressions and order
are the same: the launches of gmc_step (tiles that take the rows of short
filters through the whole stage; the polar rows in bands of whole circles, or
spread over three launches) and the three kernels that gmc_kernel_times times
on every grid."""
import ctypes as C

import numpy as np
import pytest

from gmcore_amd.capi import dptr

from gmcore_amd.host import Setup
from helpers import STATE, make_gpu, make_oracle, namelist, rel_err, seeded_ic

pytestmark = pytest.mark.gpu

# columns and rows that fill the tendency kernel's 60 x 11 tiles exactly, by one
# column pair or row more or less, or not even once
GRIDS = [(8, 5), (16, 11), (58, 12), (60, 22), (62, 23), (64, 33), (118, 34), (120, 61), (122, 66)]


@pytest.mark.parametrize("scheme", ["pc2", "wrfrk3"])
@pytest.mark.parametrize("nlon,nlat", GRIDS)
def test_stage_on_tile_edges(nlon, nlat, scheme):
    st = Setup(namelist(nlon, nlat, dt=min(600.0, 20000.0 / max(nlon, nlat)), time_scheme=scheme))
    ic = seeded_ic(st, lmax=4, seed=nlon)
    o, g = make_oracle(st, ic), make_gpu(st, ic)
    o.prepare(1)
    g.prepare(1)
    o.step(st.nl.dt_dyn, 2)
    g.step(2)
    for f in STATE + ("u_f", "v_f"):
        assert rel_err(g.download(g.level, f), o.get(o.level, f)) <= 1e-12, f


# the narrowest and lowest grids of the tiles, and the first below each; odd
# and even zones; the widest circles of the bands and the first beyond; wide
# filters (long steps) and none (short ones)
FORMS = [(62, 30, 1.0), (64, 23, 1.0), (64, 24, 1.0), (66, 25, 3.0), (108, 61, 1.0), (110, 60, 2.0), (180, 91, 5.0),
         (502, 64, 1.0), (516, 65, 4.0), (560, 64, 1.0), (602, 127, 3.0), (722, 100, 0.2),
         # circles too wide for LDS: the tiles shared out from 640 tiles on
         (602, 638, 1.0), (602, 640, 1.0), (722, 601, 0.2), (1442, 300, 3.0)]


@pytest.mark.parametrize("nlon,nlat,long", FORMS)
@pytest.mark.parametrize("option", ["plain", "stokes off, coriolis 2", "midpoint", "tvd"])
def test_stage_forms_bitwise(nlon, nlat, long, option):
    kw = {"plain": {}, "stokes off, coriolis 2": dict(pv_pole_stokes=False, coriolis_scheme=2),
          "midpoint": dict(pv_scheme="midpoint"), "tvd": dict(pv_scheme="tvd")}[option]
    st = Setup(namelist(nlon, nlat, dt=20000.0 * long / max(nlon, nlat), **kw))
    ic = seeded_ic(st, lmax=4, seed=nlon)
    a, b = make_gpu(st, ic), make_gpu(st, ic)
    for m in (a, b):
        m.prepare(1)
        m.keep_derived()    # the taping variant (pv here, the others through the sums of diagnose)
    a.step(2)
    kt, nk = np.zeros(8), C.c_int32()
    assert b.lib.gmc_kernel_times(b.ctx, st.nl.dt_dyn, 2, dptr(kt), 8, C.byref(nk)) == 0
    for level in (1, 2, 3):
        for f in STATE + ("u_f", "v_f", "gz_f", "pv"):
            np.testing.assert_array_equal(a.download(level, f), b.download(level, f), err_msg=f"{level} {f}")
    assert np.array_equal(a.diagnose(), b.diagnose())
    for m in (a, b):
        m.keep_derived(False)
    a.step(3)
    assert b.lib.gmc_kernel_times(b.ctx, st.nl.dt_dyn, 3, dptr(kt), 8, C.byref(nk)) == 0
    for f in STATE + ("u_f", "v_f", "gz_f"):
        np.testing.assert_array_equal(a.download(a.level, f), b.download(b.level, f), err_msg=f)
