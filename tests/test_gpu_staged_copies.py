"""The drop-in calls' copies, staged in pinned memory and per field: the columns of
the filter's range come back as the oracle computes them and the others untouched.

Each test prints its case before the GPU work starts.
"""
import numpy as np
import pytest

from ctsm_amd import abi, synthetic as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


STAGED_BYTES = 128 << 20    # the largest copy the library stages (kStageBytes)


def fields_bytes(st, filt):
    """What the column fields of the filter's range take packed, each to 256 bytes."""
    w = int(filt.max()) - int(filt.min()) + 1
    row = [(st.col[n].size // st.dims.ncol) * w * st.col[n].itemsize for n, _, _ in abi.COL_FIELDS]
    return sum(-(-b // 256) * 256 for b in row)


# 40,000 columns exceed the staged size, the smaller ones do not; the second call of a
# pair finds the staging, or the copies per field, of the first
@pytest.mark.parametrize("sizes", [(1, 300), (300, 1024), (40000, 300), (300, 40000)])
def test_range_of_columns_bitwise(ctx, sizes):
    for ncol in sizes:
        st = S.workload("uneven", ncol=ncol)
        filt = np.arange(ncol, 1 + ncol // 3, -2, dtype=np.int32) if ncol > 1 else np.array([1], dtype=np.int32)
        print(f"case: drop-in SoilWater, {len(filt)} of {ncol} columns", flush=True)
        assert (fields_bytes(st, filt) > STAGED_BYTES) == (ncol == 40000)
        g = st.copy()
        for f in ("smp_l", "qout", "num_substeps"):
            g.col[f][...] = st.col[f][...] = -7.0
        ctx.soilwater(g, filter_=filt)
        assert O.soilwater(st, filter_=filt)[0] == 0
        for f, v in st.col.items():
            np.testing.assert_array_equal(g.col[f], v, err_msg=f)
