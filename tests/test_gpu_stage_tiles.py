"""The fused stage at the edges of its tiles: grids whose columns and rows
fill the tendency kernel's 60 x 11 tiles exactly, by one column pair or row
more or less, or not even once.  Bar: 1e-12 relative against the oracle (the
per-step bar of the SW fields: both evaluate the same expressions, only pole
sums may differ in order)."""
import pytest

from gmcore_amd.host import Setup
from helpers import STATE, make_gpu, make_oracle, namelist, rel_err, seeded_ic

pytestmark = pytest.mark.gpu

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
