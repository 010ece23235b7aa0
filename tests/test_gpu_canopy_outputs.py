"""CanopyFluxes with output arrays that a caller does not want pointed at one array:
the outputs that have arrays of their own are the same, bit for bit.

Each test prints its case before the GPU work starts.
"""
import ctypes as C

import numpy as np
import pytest

from ctsm_amd import abi, synthetic as S
from ctsm_amd.state import CANOPY_ALIAS, DeviceState

pytestmark = pytest.mark.gpu

# read before they are written, so they have arrays of their own
INOUT = {"displa", "z0mv", "t_veg", "t_stem", "snocan", "liqcan", "cgrnds", "cgrndl", "gs_mol"}
FIRST_OUTPUT = "z0hv"       # the patch fields before it are inputs or INOUT


def _patch_outputs():
    names = [n for n, t, kind in abi.CANOPY_FIELDS if t == "f64" and kind == "p"]
    return [n for n in names[names.index(FIRST_OUTPUT):] if n not in INOUT and n not in CANOPY_ALIAS]


def _run(ctx, st, call, dumped=()):
    ds = DeviceState(st, ctx)
    dump = ctx.alloc(st.dims.npatch * 8)
    try:
        can = ds.canopy_struct()
        for name in dumped:
            setattr(can, name, C.cast(C.c_void_p(dump), abi._CT["f64"]))
        ds.canopy_struct = lambda: can
        call(ds)
        ctx.sync()
        return ds.to_host()
    finally:
        ctx.free(dump)
        ds.free()


def _check(ctx, st, call, half, own=()):
    dumped = [n for n in _patch_outputs()[half::2] if n not in own]
    full = _run(ctx, st, call)
    part = _run(ctx, st, call, dumped)
    for grp in ("col", "pch", "can"):
        for k, v in getattr(full, grp).items():
            if k not in dumped:
                np.testing.assert_array_equal(getattr(part, grp)[k], v, err_msg=f"{grp}.{k}")


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("first", [6, 41])       # in rounds, in one pass
@pytest.mark.parametrize("stomatal", [1, 2])
def test_unwanted_outputs_in_one_array(half, first, stomatal):
    from ctsm_amd.lib import Context, default_config
    ctx = Context(default_config(stomatalcond_method=stomatal))
    try:
        ctx.set_canopy_params(S.canopy_params(), S.pft_table())
        ctx.set_tuning(canopy_first_iterations=first)
        st = S.canopy_workload("canopy_uneven", ncol=300)
        print(f"case: CanopyFluxes, half {half} of the outputs in one array, first={first}, "
              f"stomatal={stomatal}, {st.dims.npatch} patches", flush=True)
        _check(ctx, st, ctx.canopyfluxes_dev, half)
    finally:
        ctx.close()


@pytest.mark.parametrize("half", [0, 1])
def test_unwanted_outputs_in_one_array_phs(half):
    from ctsm_amd import phs as PH
    from ctsm_amd.lib import Context, default_config
    npft = len(S.pft_table()["dleaf"])
    ctx = Context(default_config(use_hydrstress=1))
    try:
        ctx.set_canopy_params(S.canopy_params(), S.pft_table())
        ctx.set_phs_params(PH.default_params(npft, (np.arange(npft) >= 15).astype(np.float64)))
        st = S.canopy_workload("canopy_uneven", ncol=100)
        A = PH.canopy_phs(st, 5)
        print(f"case: CanopyFluxes PHS, half {half} of the outputs in one array, {st.dims.npatch} patches", flush=True)

        def call(ds):
            dphs = PH.DeviceCanopyPhs(ctx, A, ds)
            ctx.canopyfluxes_phs_dev(ds, dphs)
            ctx.sync()
            dphs.free()

        # the hydraulics' own results pass through qflx_tran_veg
        _check(ctx, st, call, half, own=("qflx_tran_veg",))
    finally:
        ctx.close()
