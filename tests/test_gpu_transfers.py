"""Field transfers through the pinned stage: fields of one piece, of several
and of enough for the helper threads, packed and with a leading dimension
beyond the columns, down to one row.  Bar: every value comes back as it went."""
import ctypes as C

import numpy as np
import pytest

from gmcore_amd.baro import Baroclinic
from gmcore_amd.capi import BARO_FIELD, dptr
from gmcore_amd.host import Mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlon,nlat,nlev,pad", [(16, 9, 2, 0), (16, 9, 2, 5), (362, 181, 2, 0), (360, 181, 4, 0),
                                                (360, 181, 10, 3), (360, 181, 32, 0),
                                                # two pieces of 2 MB just not and just reached, three
                                                (512, 256, 3, 0), (512, 257, 4, 0), (512, 257, 6, 0)])
def test_fields_come_back(nlon, nlat, nlev, pad):
    mesh = Mesh(nlon, nlat, 6371220.0, 7.292e-5)
    b = Baroclinic(mesh, np.linspace(0.0, 1.0, nlev + 1) * 0.1, np.linspace(0.0, 0.9, nlev + 1))
    rng = np.random.default_rng(nlon + nlev)
    for name in ("pt", "ph_lev", "v_f", "phs"):
        levels, rows, _ = b.shape(name)
        a = rng.standard_normal((levels * rows, nlon + pad))
        back = np.full_like(a, -7.0)
        assert b.lib.gmc_baro_set(b.h, BARO_FIELD[name], dptr(a), nlon + pad) == 0
        for _ in range(2):      # the stage's second use
            assert b.lib.gmc_baro_get(b.h, BARO_FIELD[name], dptr(back), nlon + pad) == 0
            np.testing.assert_array_equal(back[:, :nlon], a[:, :nlon])
            assert (back[:, nlon:] == -7.0).all()
