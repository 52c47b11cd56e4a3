"""The fused stage kernels divide by row metric terms (cell and vertex areas,
edge lengths) and by gravity through div_rn (gmcore_amd/csrc/gmc_arith.hpp): the
quotient from the correctly rounded reciprocal plus one fma correction.  The
advection kernels divide by 3 and 6, and for several tracers by Courant numbers,
areas and masses, the same way; pv and the tangential winds divide by depths
through div_mid, whose reciprocal is two Newton steps from the hardware's
estimate, and the upwind weights through div_root, with a root from an estimate
as well.  The kernels stay bit-identical to the oracle only if these give the IEEE results.  This test
compiles the header's own code for the host, the hardware's estimates replaced
by exact ones with an error of up to 2^-22, and checks it against the host's
quotients and roots: for every divisor of four real meshes (and adversarial
divisors) with random numerators and numerators whose quotient lies next to a
rounding midpoint, and for roots next to midpoints.  That the hardware's
estimates are as good is checked by the parity tests on the GPU.
"""
import os
import subprocess

import numpy as np
import pytest

from gmcore_amd.host import Setup
from gmcore_amd.namelist import Namelist

HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
def test_div_rn_equals_ieee_quotient(tmp_path):
    from gmcore_amd import capi
    src = __file__.replace("test_div_rn.py", "native/div_rn_check.cpp")
    exe = tmp_path / "div_rn_check"
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-o", str(exe), src],
                   check=True)
    fields = [capi.MESH_FIELDS.index(f) for f in ("area_cell", "area_vtx", "de_lon", "de_lat")]
    divisors = [9.80616, 3.0, 6.0]   # gravity; the PPM divisors of the advection kernels
    for nlon, nlat in ((72, 37), (180, 91), (360, 181), (1440, 721)):
        met = Setup(Namelist(num_lon=nlon, num_lat=nlat)).mesh.metrics
        for f in fields:
            divisors.extend(met[f].ravel().tolist())
    d = np.unique(np.asarray(divisors, dtype=np.float64))
    (tmp_path / "d.bin").write_bytes(d.tobytes())
    r = subprocess.run([str(exe), str(tmp_path / "d.bin"), "2000", "7"], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert "mismatches 0" in r.stdout
