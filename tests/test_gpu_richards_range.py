"""The Richards solve where its operands leave the range in which a reciprocal gives an
IEEE quotient, bit for bit against the oracle: no soil has such parameters, but the
entry points take them.

Each test prints its case before the GPU work starts.
"""
import numpy as np
import pytest

from ctsm_amd import synthetic as S
from ctsm_amd.lib import CtsmError
from helpers import soil_mask
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NCOL = 200


def faint_flux(st):
    """Conductivities down to the subnormals, over layers of 1e-6 of their thickness: the
    remainders of the fluxes' divisions are below the smallest subnormal."""
    st.col["hksat"] *= 10.0 ** np.linspace(-260.0, -312.0, NCOL)
    for k in ("dz", "z", "h2osoi_liq", "h2osoi_ice"):
        st.col[k] *= 1e-6


def thin(st):
    """Layers of 1e-149 to 1e-130 m: diagonals of 2^1000 and below."""
    f = 10.0 ** np.linspace(-149.0, -130.0, NCOL)
    for k in ("dz", "z", "h2osoi_liq"):
        st.col[k] *= f
    st.col["h2osoi_ice"][...] = 0.0


def steep(st):
    """Retention exponents up to 110 over nearly dry layers."""
    st.col["bsw"][...] = np.linspace(20.0, 110.0, NCOL)
    st.col["h2osoi_liq"] *= 0.02


def trickle(st):
    """No conductivity, and an infiltration down to the subnormals on dry layers."""
    st.col["hksat"][...] = 0.0
    st.col["qflx_rootsoi"][...] = 0.0
    st.col["h2osoi_liq"][...] = 0.0
    st.col["qflx_infl"][...] = 10.0 ** np.linspace(-322.0, -270.0, NCOL)


def solved_by_oracle(st):
    """The oracle's state, column by column, and the columns it solves."""
    o = st.copy()
    ok = [O.soilwater(o, filter_=np.array([c], dtype=np.int32))[0] == 0 for c in range(1, NCOL + 1)]
    return o, np.array(ok)


def check(ctx, st, lanes):
    before = ctx.get_tuning()
    ctx.set_tuning(richards_lanes=lanes, richards_block=64)
    o, ok = solved_by_oracle(st)
    assert ok.sum() > NCOL // 2
    g = st.copy()
    try:
        ctx.soilwater(g)
        assert ok.all()
    except CtsmError as e:
        assert not ok[e.index - 1]
    finally:
        ctx.set_tuning(**before)
    m = soil_mask(st) & ok
    for f in ("smp_l", "hk_l", "qin", "qout"):
        np.testing.assert_array_equal(np.where(m, g.col[f], 0.0), np.where(m, o.col[f], 0.0), err_msg=f)
    for f in ("h2osoi_liq", "qcharge", "num_substeps"):
        np.testing.assert_array_equal(np.where(ok, g.col[f], 0.0), np.where(ok, o.col[f], 0.0), err_msg=f)


@pytest.mark.parametrize("lanes", [0, 4, 8])
@pytest.mark.parametrize("change", [faint_flux, thin, steep, trickle])
def test_beyond_the_range_bitwise(ctx, change, lanes):
    st = S.workload("uneven", ncol=NCOL)
    change(st)
    print(f"case: SoilWater, {change.__name__}, {lanes} lanes", flush=True)
    check(ctx, st, lanes)


def nan_at_the_bottom(st):
    """A retention exponent that is NaN in the last layer of every fourth column, beside
    columns beyond the range."""
    nb = st.col["nbedrock"]
    nb[::2] = 20
    st.col["bsw"][:, 1::2] = 30.0
    st.col["bsw"][nb[::4] - 1, np.arange(0, NCOL, 4)] = np.nan


def flood(st):
    """Infinite infiltration into every third column."""
    st.col["qflx_infl"][::3] = np.inf


@pytest.mark.parametrize("lanes", [0, 4, 8])
@pytest.mark.parametrize("change", [nan_at_the_bottom, flood])
def test_nan_and_infinity_bitwise(ctx, change, lanes):
    st = S.workload("uneven", ncol=NCOL)
    change(st)
    print(f"case: SoilWater, {change.__name__}, {lanes} lanes", flush=True)
    check(ctx, st, lanes)
