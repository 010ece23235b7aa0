"""Runs one case of test_gpu_refused_memory.py: child.py <refuse.so> <case>."""
import ctypes as C
import sys

shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)      # before the library

import numpy as np  # noqa: E402

from ctsm_amd import synthetic as S  # noqa: E402
from ctsm_amd.lib import Context  # noqa: E402
from ctsm_amd.state import DeviceState  # noqa: E402
from oracle import oracle as O  # noqa: E402

shim.refuse_device.argtypes = shim.refuse_pinned.argtypes = [C.c_size_t, C.c_size_t]


def same(a, b):
    for grp in ("col", "pch", "can"):
        for k, v in getattr(b, grp).items():
            np.testing.assert_array_equal(getattr(a, grp)[k], v, err_msg=f"{grp}.{k}")


def one_pass_context(plain):
    ctx = Context()
    ctx.set_canopy_params(S.canopy_params(), S.pft_table())
    ctx.set_tuning(**(dict(plain_routines=1) if plain else dict(canopy_first_iterations=41)))
    return ctx


def one_pass(plain, graph):
    """CanopyFluxes without rounds where the device has an eighth of the work buffer."""
    st = S.canopy_workload("canopy_uneven", ncol=501)
    work = 128 * st.dims.npatch
    print(f"case: one-pass CanopyFluxes, {st.dims.npatch} patches, plain={plain}, graph={graph}, "
          f"{work} bytes of work refused", flush=True)
    results = []
    for refuse in (False, True):
        ctx = one_pass_context(plain)
        ds = DeviceState(st, ctx)
        if refuse:
            shim.refuse_device(work // 8, work)
        if graph:
            g = ctx.graph_capture(ds, nsteps=1, canopy=True)
            shim.refuse_device(0, 0)
            for _ in range(2):
                ctx.graph_launch(g)
                ctx.sync()
            ctx.graph_destroy(g)
        else:
            for _ in range(2):
                ctx.canopyfluxes_dev(ds)
            ctx.sync()
            shim.refuse_device(0, 0)
        assert (shim.refusals() > 0) == refuse
        results.append(ds.to_host())
        ds.free()
        ctx.close()
    same(results[1], results[0])


def host_arrays(what):
    """SoilWater on host arrays: no pinned memory at all, none on a call that needs more
    than the one before it, or no device memory for the fields in one piece; every call
    right, and the copies in one piece again once there is memory."""
    ctx = Context()
    print(f"case: SoilWater on host arrays, no memory: {what}", flush=True)
    for ncol, full in ((300, what != "pinned later"), (2000, True), (700, False)):
        if full:
            size = 2000 * ncol      # less than the fields take in one piece, more than one takes
            if what == "device":
                shim.refuse_device(size, 1 << 40)
            else:
                shim.refuse_pinned(0, 1 << 40)
        st = S.workload("uneven", ncol=ncol)
        g = st.copy()
        ctx.soilwater(g)
        shim.refuse_device(0, 0)
        shim.refuse_pinned(0, 0)
        assert (shim.refusals() > 0) == full, ncol
        assert O.soilwater(st)[0] == 0
        for k, v in st.col.items():
            np.testing.assert_array_equal(g.col[k], v, err_msg=f"{ncol} columns: {k}")
    ctx.close()


CASES = {
    "host_arrays_pinned": lambda: host_arrays("pinned"),
    "host_arrays_pinned_later": lambda: host_arrays("pinned later"),
    "host_arrays_device": lambda: host_arrays("device"),
    "one_pass": lambda: one_pass(False, False),
    "one_pass_plain": lambda: one_pass(True, False),
    "one_pass_graph": lambda: one_pass(False, True),
}

if __name__ == "__main__":
    CASES[sys.argv[2]]()
    print("same", flush=True)
