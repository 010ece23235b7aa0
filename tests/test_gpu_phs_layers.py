"""calcstress with the soil staged in LDS at the edges of its layer count (the
fewest layers a context takes, a partial set, all of them) and of its blocks
(one patch short of and past a wavefront), bit for bit against the oracle."""
import numpy as np
import pytest

from ctsm_amd import phs as PH
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlevsoi", [2, 13, 19, 20])
@pytest.mark.parametrize("ncol", [63, 65])
def test_calcstress_layers(nlevsoi, ncol):
    from ctsm_amd.lib import Context, default_config
    print(f"case: calcstress, {nlevsoi} soil layers, {ncol} patches", flush=True)
    ctx = Context(default_config(nlevsoi=nlevsoi))
    try:
        ctx.set_phs_params(PH.default_params())
        A = PH.synthetic_stress(ncol, max_patches=1, seed=nlevsoi, nlevsoi=nlevsoi)
        ref = A.copy()
        assert O.phs_calcstress(ref, PH.default_params()) == 0
        ctx.phs_calcstress(A.layout(), A.host_struct(), A.npatch)
        for k in ("vegwp", "vegwp_pd", "bsun", "bsha", "qflx_tran_veg"):
            np.testing.assert_array_equal(A[k], ref[k], err_msg=k)
    finally:
        ctx.close()
