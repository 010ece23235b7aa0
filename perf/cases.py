"""The work this library's users have it do, as cases that can be timed and checked.

A case is one call (or one captured graph of calls) of the public entry points
on a seeded synthetic state:

  land     the full land step in clm_drv order (CanopyFluxes, SoilTemperature,
           SoilFluxes, the sink, the surface water, SoilWater, the water tables,
           the drainage) on device-resident state, eager or as a graph
  canopy   CanopyFluxes alone, over all patches or a filter of them
  phs      CanopyFluxes with plant hydraulic stress
  soil     soil steps (SoilTemperature, SetSoilWaterFractions, SoilWater) of a
           batch without patches to speak of, captured as one graph
  water    SoilWater (the Richards solve) alone
  heat     SoilTemperature alone
  stress   calcstress (the Newton solve of the vegetation water potential)
  history  one step of the default history tape
  dropin   the three soil routines on host arrays, as a Fortran host calls them

Sizes and distributions are those of ctsm_amd.synthetic: 1-16 patches per
column, snow of 0-12 layers and bedrock at 5-20 layers where `snow` is set.
Batches above TILE columns repeat one generated tile of at most TILE columns,
stored in binned (snow, bedrock) order as the batched entries are meant to be fed.
"""
import math

import numpy as np
import torch

from ctsm_amd import abi, lib, phs, synthetic
from ctsm_amd.history import DEFAULT_FIELDS, HistoryTape
from ctsm_amd.state import CANOPY_ALIAS, SOILFLUX_OWN, DeviceState

DTIME = 1800.0
TILE = 65536
NPFT = len(synthetic.pft_table()["dleaf"])
CROP = (np.arange(NPFT) >= 15).astype(np.float64)
# means of the generated distributions, for work(): patches per column, snow
# layers, bedrock index (Richards layers)
PATCHES, SNOW, BEDROCK = 8.5, 6.0, 12.5


def listed():
    land = {"kind": "land", "stomata": "medlyn", "biomass": True}
    canopy = {"kind": "canopy", "stomata": "medlyn", "z0": "meier", "biomass": True, "share": 1.0}
    return [
        # a small ensemble member served alone: latency and launches count
        dict(land, name="land_300", ncol=300, snow=False, graph=False),
        # a region or a pool of members, stepped eagerly
        dict(land, name="land_20000", ncol=20000, snow=True, graph=False),
        # one GPU's share of a 1/8 degree grid, the step captured once and replayed
        dict(land, name="land_1048576", ncol=1048576, snow=True, graph=True),
        # CanopyFluxes by itself on every patch, the default namelist
        dict(canopy, name="canopy_65536", ncol=65536, snow=True),
        # the older namelist (Ball-Berry, Zeng-Wang roughness, no biomass heat) on the
        # exposed-vegetation filter of an odd-sized domain
        dict(canopy, name="canopy_bb_8191", ncol=8191, snow=False, stomata="ballberry", z0="zengwang", biomass=False,
             share=0.7),
        # the hydraulic-stress configuration, day and night patches
        {"name": "phs_4096", "kind": "phs", "ncol": 4096, "snow": True, "stomata": "medlyn"},
        # the batched uneven soil columns: eight steps in one graph
        {"name": "soil_65536", "kind": "soil", "ncol": 65536, "snow": True, "steps": 8},
        # the two solves alone, at a quarter of the large grid
        {"name": "water_262144", "kind": "water", "ncol": 262144, "snow": True},
        {"name": "heat_262144", "kind": "heat", "ncol": 262144, "snow": True},
        # vegetation water potentials, one patch per column
        {"name": "stress_262144", "kind": "stress", "ncol": 262144},
        # accumulating the default 15-field tape every step
        {"name": "history_262144", "kind": "history", "ncol": 262144, "snow": True},
        # a Fortran host keeping its own arrays, one clump of columns per call
        {"name": "dropin_1024", "kind": "dropin", "ncol": 1024, "snow": False},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["land", "land", "land", "canopy", "canopy", "phs", "soil", "water", "heat", "stress",
                       "history", "dropin"])
    c = {"kind": kind}
    if kind != "stress":
        c["snow"] = rng.random() < 0.6
    if kind == "land":
        c.update(ncol=_size(rng, 64, 400000), graph=rng.random() < 0.5, stomata=rng.choice(["medlyn", "ballberry"]),
                 biomass=rng.random() < 0.7)
        c["snow"] = c["snow"] and c["ncol"] >= 16384
    elif kind == "canopy":
        c.update(ncol=_size(rng, 64, 300000), stomata=rng.choice(["medlyn", "ballberry"]),
                 z0=rng.choice(["meier", "zengwang"]), biomass=rng.random() < 0.7,
                 share=rng.choice([1.0, 1.0, 0.7, 0.2]))
    elif kind == "phs":
        c.update(ncol=_size(rng, 64, 16384), stomata=rng.choice(["medlyn", "ballberry"]))
    elif kind == "soil":
        c.update(ncol=_size(rng, 256, 262144), steps=rng.choice([1, 2, 4, 8]))
    elif kind in ("water", "heat"):
        c.update(ncol=_size(rng, 256, 1000000))
    elif kind == "stress":
        c.update(ncol=_size(rng, 256, 262144))
    elif kind == "history":
        c.update(ncol=_size(rng, 1024, 262144))
    else:
        c.update(ncol=_size(rng, 16, 8192))
    if kind != "stress":        # a large batch repeats one tile
        c["ncol"] = _tile(c["ncol"]) * -(-c["ncol"] // TILE)
    return c


# ---- contexts and states -----------------------------------------------------

_contexts = {}


def _context(case):
    """The program's library context for this namelist, made once and kept."""
    kw = {}
    if case["kind"] in ("land", "canopy", "phs"):
        kw = {"stomatalcond_method": 2 if case["stomata"] == "medlyn" else 1,
              "z0param_method": 0 if case.get("z0") == "zengwang" else 1,
              "use_biomass_heat_storage": int(case.get("biomass", True)),
              "use_hydrstress": int(case["kind"] == "phs")}
    key = tuple(sorted(kw.items()))
    if key not in _contexts:
        ctx = lib.Context(lib.default_config(**kw))
        ctx.set_canopy_params(synthetic.canopy_params(), synthetic.pft_table())
        ctx.set_phs_params(phs.default_params(NPFT, CROP))
        _contexts[key] = ctx
    return _contexts[key]


def _tile(ncol):
    """Columns generated for a batch of ncol: all, or the equal parts it repeats."""
    return ncol // -(-ncol // TILE)


def _host(case, seed):
    """The generated state: the whole batch, or the tile that it repeats.  A column
    has 1-16 patches, each count equally often for every seed."""
    n = _tile(case["ncol"])
    vegetated = case["kind"] in ("land", "canopy", "phs", "history")
    ids = np.arange(n, dtype=np.int64)
    if vegetated:
        some = np.arange(2 * n + 1024, dtype=np.int64)
        count = np.floor(synthetic.uniform(seed, synthetic.S_NPATCH, some) * 16).astype(np.int64)
        by_count = some[np.argsort(count, kind="stable")]
        start = np.concatenate([[0], np.cumsum(np.bincount(count, minlength=16))])
        ids = np.sort(np.concatenate([by_count[start[k]:start[k] + (n + 15 - k) // 16] for k in range(16)]))
        assert len(ids) == n
    nsno, nbed = synthetic.structure(int(ids.max()) + 1, seed, snow=case["snow"], bedrock=case["snow"])
    ids = ids[np.lexsort((nbed[ids], nsno[ids]))]
    if vegetated:
        return synthetic.canopy_workload("canopy_uneven" if case["snow"] else "canopy", seed=seed, gids=ids)
    return synthetic.soil_only(n, seed, snow=case["snow"], bedrock=case["snow"], gids=ids)


class _Memory:
    """Device memory of one state.  The state and every tensor that views the
    memory hold this object; it is given back when the last of them goes."""

    def __init__(self, ctx):
        self.ctx, self.held, self.graph = ctx, [], None

    def __del__(self):
        try:
            self.ctx.sync()
            if self.graph is not None:
                self.ctx.graph_destroy(self.graph)
            for x in self.held:
                if isinstance(x, int):
                    self.ctx.free(x)
                else:
                    x.free()
        except Exception:       # at the interpreter's end the library may be gone already
            pass


class _Raw:
    def __init__(self, memory, ptr, shape, dtype):
        self.memory = memory
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(int(s) for s in shape),
                                         "typestr": np.dtype(dtype).str, "version": 2}


def _tensor(memory, ptr, shape, dtype):
    """A torch view of device memory that the library allocated (the view holds
    the _Raw, and with it the memory)."""
    return torch.as_tensor(_Raw(memory, ptr, shape, dtype), device="cuda")


_PATCH_KIND = {"p", "soip", "lyr"}
_CANOPY_KIND = {n: k for n, _, k in abi.CANOPY_FIELDS}
_SOILFLUX_KIND = {n: k for n, _, k in SOILFLUX_OWN}


class _Tiled(DeviceState):
    """A DeviceState of ncol columns that repeats a host state's columns."""

    def __init__(self, host, ctx, ncol):
        self.ctx = ctx
        base, self._shapes = host.dims, {}
        self.col, self.pch, self.can, self.sf, self.hy = {}, {}, {}, {}, {}
        times = ncol // base.ncol
        npatch = times * base.npatch
        self.dims = type(base)(ncol, npatch, base.nlevsno, base.nlevsoi, base.nlevgrnd, ncol if base.ngrid else 0)
        shift = {("c", "patchi"): base.npatch, ("c", "patchf"): base.npatch, ("p", "column"): base.ncol,
                 ("g", "gridcell"): base.ncol}
        for group, src, dst in (("c", host.col, self.col), ("p", host.pch, self.pch), ("g", host.can, self.can),
                                ("s", host.sf, self.sf), ("y", host.hy, self.hy)):
            for k, a in src.items():
                patch = (group == "p" or (group == "g" and _CANOPY_KIND[k] in _PATCH_KIND)
                         or (group == "s" and _SOILFLUX_KIND[k] == "p"))
                n, b = (npatch, base.npatch) if patch else (ncol, base.ncol)
                shape = a.shape[:-1] + (n,)
                dst[k] = ctx.alloc(max(int(np.prod(shape)) * a.itemsize, 8))
                self._shapes[(group, k)] = (shape, a.dtype)
                out, one = _tensor(self, dst[k], shape, a.dtype), torch.from_numpy(np.ascontiguousarray(a)).cuda()
                step = shift.get((group, k), 0)
                for i in range(times):
                    out[..., i * b:(i + 1) * b] = one + i * step if step else one
        torch.cuda.synchronize()


class State:
    """What the caller's program holds: the context, the device state and, where
    a case restarts from the same state each pass, a copy of what it changes."""

    def __init__(self, case, ctx, ds=None):
        self.case, self.ctx, self.ds, self.memory = case, ctx, ds, _Memory(ctx)
        self.graph = self.tape = self.arrays = None
        self.saved, self.outputs = [], {}
        if isinstance(ds, DeviceState):
            self.memory.held.append(ds)

    def hold(self, thing):
        """A device pointer, or an object with free(), that goes with the state."""
        self.memory.held.append(thing)
        return thing

    def keep(self, group, name):
        """Restore this field before each pass."""
        ptr = getattr(self.ds, {"c": "col", "g": "can"}[group])[name]
        shape, dt = self.ds._shapes[(group, name)]
        self.keep_raw(ptr, int(np.prod(shape)) * np.dtype(dt).itemsize)

    def keep_raw(self, ptr, nbytes):
        copy = self.hold(self.ctx.alloc(nbytes))
        self.ctx.copy(copy, ptr, nbytes)
        self.saved.append((ptr, copy, nbytes))

    def restore(self):
        for dst, src, nbytes in self.saved:
            self.ctx.copy(dst, src, nbytes)

    def view(self, ptr, shape, dtype):
        return _tensor(self.memory, ptr, shape, dtype)

    def views(self, group, names):
        """Tensors over fields of the device state, aliases resolved."""
        ds, out = self.ds, {}
        for n in names:
            g, k = group, n
            if group == "g" and n in CANOPY_ALIAS:
                g, k = CANOPY_ALIAS[n]
            elif group == "y" and n == "qflx_infl":
                g = "c"
            ptr = {"c": ds.col, "p": ds.pch, "g": ds.can, "s": ds.sf, "y": ds.hy}[g][k]
            out[n] = self.view(ptr, *ds._shapes[(g, k)])
        return out


_COL_OUT = ("t_soisno", "h2osoi_liq", "h2osoi_ice", "t_grnd", "h2osfc", "eflx_fgr", "thk", "imelt")
_WATER_OUT = ("h2osoi_liq", "smp_l", "hk_l", "qin", "qout", "qcharge", "num_substeps")
_HEAT_OUT = ("t_soisno", "h2osoi_liq", "h2osoi_ice", "t_h2osfc", "t_grnd", "thk", "fact", "eflx_fgr", "imelt",
             "qflx_snomelt", "xmf")
_CANOPY_OUT = ("t_veg", "t_stem", "liqcan", "snocan", "displa", "z0mv", "taf", "qaf", "ustar", "um", "obu", "rb1",
               "rah1", "rah2", "btran", "rootr", "psnsun", "psnsha", "fpsn", "gs_mol_sun", "gs_mol_sha", "cisun_z",
               "rssun", "rssha", "lmrsun", "qflx_tran_veg", "qflx_evap_veg", "eflx_sh_veg", "eflx_sh_grnd",
               "qflx_evap_soi", "cgrnd", "t_ref2m", "rh_ref2m", "u10", "vds", "ulrad", "dlrad", "taux", "t_skin",
               "num_iter", "rh_af", "kc", "vcmax_z")
_LAND_OUT = {"c": _COL_OUT + ("qout", "qflx_rootsoi"),
             "g": ("t_veg", "t_stem", "liqcan", "taf", "qaf", "ustar", "obu", "btran", "rootr", "fpsn", "gs_mol_sun",
                   "gs_mol_sha", "qflx_tran_veg", "qflx_evap_veg", "eflx_sh_veg", "t_ref2m", "rh_ref2m", "u10",
                   "ulrad", "num_iter", "z0mv"),
             "s": ("eflx_sh_tot", "eflx_lh_tot", "eflx_soil_grnd", "eflx_lwrad_out"),
             "y": ("qflx_infl", "qflx_surf", "zwt", "zwt_perched", "frost_table", "h2osoi_vol", "qflx_drain",
                   "qflx_runoff")}


def prepare(case, seed):
    kind, ctx = case["kind"], _context(case)
    if kind == "stress":
        a = phs.synthetic_stress(case["ncol"], max_patches=1, seed=seed)
        s = State(case, ctx)
        s.arrays = s.hold(phs.DevicePhs(ctx, a))
        s.layout, s.struct, s.npatch = a.layout(), s.arrays.struct(), a.npatch
        s.keep_raw(s.arrays.ptr["vegwp"], a["vegwp"].nbytes)
        s.outputs = {k: s.view(s.arrays.ptr[k], a[k].shape, a[k].dtype)
                     for k in ("vegwp", "bsun", "bsha", "qflx_tran_veg")}
        ctx.sync()
        return s
    host = _host(case, seed)
    if kind == "dropin":
        s = State(case, ctx, host)
        s.first = {k: host.col[k].copy() for k in ("t_soisno", "h2osoi_liq", "h2osoi_ice")}
        s.outputs = {k: host.col[k] for k in dict.fromkeys(_HEAT_OUT + _WATER_OUT)}
        return s
    canopy_phs = phs.canopy_phs(host, seed) if kind == "phs" else None
    ds = DeviceState(host, ctx) if case["ncol"] <= TILE else _Tiled(host, ctx, case["ncol"])
    s = State(case, ctx, ds)
    if kind == "land":
        s.structs = (*ds.structs(), ds.canopy_struct(), ds.soilflux_struct())
        s.hydro = synthetic.hydro_params()
        if case["graph"]:
            s.graph = s.memory.graph = ctx.graph_capture_full(ds, nsteps=1, hydro=s.hydro, water_table=True,
                                                              drainage=True, dtime=DTIME)
        for g, names in _LAND_OUT.items():
            s.outputs.update(s.views(g, names))
    elif kind == "canopy":
        s.structs = (*ds.structs(), ds.canopy_struct())
        s.filter, s.n = None, ds.dims.npatch
        if case["share"] < 1.0:
            pick = np.random.default_rng(seed).random(ds.dims.npatch) < case["share"]
            f = (np.nonzero(pick)[0] + 1).astype(np.int32)
            s.filter, s.n = ctx.device_array(f), len(f)
            s.hold(s.filter)
        if case["z0"] == "zengwang":        # CanopyTemperature sets these two before every CanopyFluxes
            s.keep("g", "displa")
            s.keep("g", "z0mv")
        s.outputs = s.views("g", _CANOPY_OUT)
    elif kind == "phs":
        s.arrays = s.hold(phs.DeviceCanopyPhs(ctx, canopy_phs, ds))
        s.keep_raw(s.arrays.ptr["vegwp"], canopy_phs["vegwp"].nbytes)
        s.outputs = s.views("g", [n for n in _CANOPY_OUT if n != "vcmax_z"])
        s.outputs.update({k: s.view(s.arrays.ptr[k], canopy_phs[k].shape, canopy_phs[k].dtype)
                          for k in ("vegwp", "bsun", "bsha", "an_sun", "an_sha", "k_soil_root")})
    elif kind == "history":
        s.tape = s.hold(HistoryTape(ctx, ds))
        for spec, d in zip(s.tape.specs, s.tape.desc):
            s.outputs[spec[0]] = (s.view(d.hbuf, (d.num2d, d.n1d), np.float64),
                                  s.view(d.nacs, (d.num2d, d.n1d), np.int32))
    else:
        for k in ("t_soisno", "h2osoi_liq", "h2osoi_ice") if kind != "water" else ("h2osoi_liq",):
            s.keep("c", k)
        if kind == "soil":
            s.graph = s.memory.graph = ctx.graph_capture(ds, nsteps=case["steps"], canopy=False,
                                                         structs=(*ds.structs(), None))
        s.outputs = s.views("c", {"soil": dict.fromkeys(_HEAT_OUT + _WATER_OUT), "water": _WATER_OUT,
                                     "heat": _HEAT_OUT}[kind])
    ctx.sync()
    torch.cuda.synchronize()
    return s


def run(s):
    kind, ctx, ds = s.case["kind"], s.ctx, s.ds
    if kind == "land":
        if s.graph is not None:
            ctx.graph_launch(s.graph)
        else:
            ctx.land_step_full_dev(ds, structs=s.structs, hydro=s.hydro, water_table=True, drainage=True, dtime=DTIME)
    elif kind == "dropin":
        for k, v in s.first.items():
            np.copyto(ds.col[k], v)
        ctx.soiltemperature(ds, dtime=DTIME)
        ctx.soilwater_fractions(ds)
        ctx.soilwater(ds, dtime=DTIME)
    elif kind == "history":
        s.tape.update()
    else:
        s.restore()
        if kind == "canopy":
            ctx.canopyfluxes_dev(ds, filterp_dev=s.filter, n=s.n, dtime=DTIME, structs=s.structs)
        elif kind == "phs":
            ctx.canopyfluxes_phs_dev(ds, s.arrays, dtime=DTIME)
        elif kind == "soil":
            ctx.graph_launch(s.graph)
        elif kind == "water":
            ctx.soilwater_dev(ds, dtime=DTIME)
        elif kind == "heat":
            ctx.soiltemperature_dev(ds, dtime=DTIME)
        else:
            ctx.phs_calcstress(s.layout, s.struct, s.npatch, None, dev=True)
    return s.outputs


# ---- what a pass cannot do without ----------------------------------------------

def _field_bytes(fields, written, kinds):
    per = {}
    for n, t, k in fields:
        if k in kinds:
            b = (4 if t == "i32" else 8) * (25 if k in ("soip", "soi") else 1)
            per[n] = b * (2 if n in written else 1)
    return sum(per.values())


def _water_bytes(bed):
    # per layer 10 values read and 5 written; per column the index, the infiltration, two results
    return 120 * bed + 28


def _heat_bytes(snow, patches):
    # snow layers: 6 values read, 7 and a flag written; ground levels: 12 read, 6 and a flag written;
    # patches: 15 values and an index read, sabg_lyr of the layers, 3 written; column scalars; zi(0)
    return 282 + snow * 108 + 192 + 25 * 148 + patches * (148 + (snow + 1) * 8)


def _canopy_bytes():
    """(per patch, per column): every field read or written once, those that are both twice."""
    both = {"displa", "z0mv", "t_veg", "t_stem", "snocan", "liqcan", "cgrnds", "cgrndl"}
    return _field_bytes(abi.CANOPY_FIELDS, both, ("p", "soip")), 23 * 8 + 4 + 25 * 9 * 8 + 9 * 8 + 4


# FP64 operations of one leaf-temperature iteration with both leaves' stomatal solves, and the
# iterations a patch takes on average
_ITERATION, _ITERATIONS = 3500.0, 6.2


def work(case):
    n, kind = case["ncol"], case["kind"]
    snow, bed = (SNOW, BEDROCK) if case.get("snow") else (0.0, 20.0)
    per_patch, per_col = _canopy_bytes()
    if kind == "land":
        # the solves, SoilFluxes (50 patch values, 12 column values and three profiles over snow and
        # top layer), the sink, the surface water, the water tables, the drainage
        col = (per_col + _heat_bytes(snow, PATCHES) + _water_bytes(bed) + 96 + 24 * (snow + 1) + 25 * 16 + 8
               + 38 * 8 + 4 + 56 + 960 + 120 + 1600)
        return {"bytes": n * (col + PATCHES * (per_patch + 50 * 8 + 25 * 8 + 16)),
                "flops": n * (PATCHES * _ITERATION * _ITERATIONS + 60.0 * bed * 6 + 4000)}
    if kind == "canopy":
        m = n * PATCHES * case["share"]
        return {"bytes": n * per_col + m * per_patch, "flops": m * _ITERATION * _ITERATIONS}
    if kind == "phs":
        m = n * PATCHES
        return {"bytes": n * (per_col + 5 * 160) + m * (per_patch + 25 * 24 + 30 * 8),
                "flops": m * 10 * _ITERATION * _ITERATIONS}
    if kind in ("soil", "dropin"):
        steps = case.get("steps", 1)
        return {"bytes": steps * n * (_heat_bytes(snow, 1.0) + _water_bytes(bed) + 20 * 40),
                "flops": steps * n * (60.0 * bed * 6 + 4000)}
    if kind == "water":
        return {"bytes": n * _water_bytes(bed), "flops": n * 60.0 * bed * 6}
    if kind == "heat":
        return {"bytes": n * _heat_bytes(snow, 1.0), "flops": n * 4000.0}
    if kind == "stress":
        return {"bytes": n * (16 * 8 + 20 * 8 + 8 * 11 + 16 + 40 * 8), "flops": n * 12 * 60.0 * 8}
    elems = n * (25 + 20 + 20 + 9) + 3 * n * PATCHES
    return {"bytes": elems * 32.0, "flops": elems * 2.0}


# Largest relative differences between the same routines on two libms (last-bit
# differences of log, exp and pow; 700-20,000 columns), times four and rounded up
# for the rarer columns of larger batches: a column whose Richards solve sub-steps
# most, or a layer just below freezing, may take another sub-step or iteration and
# then moves by the truncation error of that step.  Seen (2-norm, largest): land
# 1.7e-8, 9.1e-7; canopy 7.5e-10, 8.3e-8; phs 6.4e-13, 3.9e-11; eight soil steps
# 2.7e-5, 5.0e-3; water 1.6e-8, 8.2e-7; heat 1.2e-15, 9.2e-14.  The history buffers
# hold sums of the fields themselves.
_TOLERANCE = {
    "land": {"rel": 1e-6, "max": 1e-2, "differ": 1e-4},
    "canopy": {"rel": 1e-7, "max": 1e-3},
    "phs": {"rel": 1e-7, "max": 1e-3},
    "soil": {"rel": 2e-4, "max": 4e-2, "differ": 1e-4},
    "water": {"rel": 1e-6, "max": 1e-4},
    "heat": {"rel": 1e-11, "max": 1e-7, "differ": 1e-6},
    "stress": {"rel": 1e-7, "max": 1e-3},
    "dropin": {"rel": 1e-6, "max": 1e-3, "differ": 1e-4},
}


def tolerance(case):
    return _TOLERANCE.get(case["kind"], "exact")


# ---- the same results in plain numpy, where they have a form of their own ------

def exact(case, seed):
    kind = case["kind"]
    if kind == "history":
        return _exact_history(case, seed)
    if kind == "water" and case["ncol"] <= 32768:
        return _richards(_host(case, seed))
    if kind == "canopy" and case["share"] == 1.0 and case["ncol"] <= TILE:
        out = dict.fromkeys(_CANOPY_OUT)
        out.update(_roughness_and_stress(_host(case, seed), case))
        return out
    if kind == "land" and case["ncol"] <= TILE:
        out = dict.fromkeys(n for g in _LAND_OUT.values() for n in g)
        got = _roughness_and_stress(_host(case, seed), dict(case, z0="meier"))
        out.update({k: v for k, v in got.items() if k in out})
        return out
    return None


def _exact_history(case, seed):
    """One update of a zeroed tape: the field itself, counted once."""
    host = _host(case, seed)
    base, out = host.dims, {}
    for name, group, key, levels, *_ in DEFAULT_FIELDS:
        a = np.atleast_2d({"c": host.col, "g": host.can, "s": host.sf, "y": host.hy}[group][key])
        if levels is not None:
            a = a[base.nlevsno:base.nlevsno + (25 if levels[2] == "levgrnd" else 20)]
        a = np.tile(a, (1, case["ncol"] // base.ncol))
        out[name] = (a, np.ones(a.shape, np.int32))
    return out


def _roughness_and_stress(st, case):
    """The canopy's roughness and displacement height (the Meier et al. 2022 or the
    Zeng and Wang 2007 form) and the soil moisture stress of the roots."""
    c, g, ns = st.col, st.can, st.dims.nlevsno
    pft, pc = synthetic.pft_table(), st.pch["column"] - 1
    row = {k: v[g["itype"]] for k, v in pft.items()}
    lai = g["elai"] + g["esai"]
    if case["z0"] == "meier":
        lt = np.maximum(1e-5, lai)
        root = np.sqrt(7.5 * lt)
        displa = g["htop"] * (1.0 + np.expm1(-root) / root)
        lt = np.minimum(lt, row["z0v_LAImax"])
        start = row["z0v_c"] * lt * 0.25 / np.sqrt(row["z0v_Cs"] + row["z0v_Cr"] * lt * 0.5)
        u, moving = start.copy(), np.ones(len(start), bool)
        while moving.any():
            new = start * np.exp(u)
            step = np.where(moving, np.abs(new - u), 0.0)
            u = np.where(moving, new, u)
            moving &= step > 1e-4
        u = 4.0 * u / lt / row["z0v_c"]
        z0 = (g["htop"] - displa) * row["z0v_cw"] * np.exp(-0.4 * u - 1.0 + 1.0 / row["z0v_cw"])
    else:
        v = np.expm1(-np.minimum(lai, 2.0)) / np.expm1(-2.0)
        displa = v * g["displa"]
        z0 = g["z0mv"] ** v * g["z0mg"][pc] ** (1.0 - v)
    vol_ice = np.minimum(c["watsat"], c["h2osoi_ice"][ns:] / (917.0 * c["dz"][ns:]))
    eff = c["watsat"] - vol_ice
    liq = np.minimum(eff, c["h2osoi_liq"][ns:] / (1000.0 * c["dz"][ns:]))
    takes = (liq > 0.0) & (c["t_soisno"][ns:] > 273.15 - 2.0)
    smp = -c["sucsat"] * np.maximum(liq / eff, 0.01) ** -c["bsw"]
    smp = np.maximum(row["smpsc"], smp[:, pc])
    rres = np.minimum((eff / c["watsat"])[:, pc] * (smp - row["smpsc"]) / (row["smpso"] - row["smpsc"]), 1.0)
    rr = np.where(takes[:, pc], g["rootfr"] * rres, 0.0)
    btran = np.maximum(rr, 0.0).sum(axis=0)
    rootr = np.where(btran > 0.0, rr / np.where(btran > 0.0, btran, 1.0), 0.0)
    return {"displa": displa, "z0mv": z0, "btran": btran, "rootr": rootr}


def _richards(st):
    """The adaptive moisture-form Richards solve with a zero-flux bottom, every
    column's tridiagonal system as one dense solve."""
    c, ns, L = st.col, st.dims.nlevsno, 20
    n = st.dims.ncol
    top = slice(ns, ns + L)
    nb = c["nbedrock"]
    lev = np.arange(L)[:, None]
    live, bottom = lev < nb, lev == nb - 1
    ws, b, suc, sink = (c[k][:L] for k in ("watsat", "bsw", "sucsat", "qflx_rootsoi"))
    mdz, z = 1000.0 * c["dz"][top], c["z"][top]
    ice = c["icefrac"][:L]
    below = np.vstack([ice[1:], ice[-1:]])
    hkc = 10.0 ** (-6.0 * np.where(bottom, ice, 0.5 * (ice + below))) * c["hksat"][:L]
    den = np.vstack([1000.0 * np.diff(z, axis=0), np.ones((1, n))])
    out = {k: np.array(c[k]) for k in _WATER_OUT}
    liq = c["h2osoi_liq"][top].copy()
    dt, done, subs = np.full(n, DTIME), np.zeros(n), np.zeros(n)
    todo = np.arange(n)
    while todo.size:
        i = todo
        lv, bt = live[:, i], bottom[:, i]
        w, bb, m, d = ws[:, i], b[:, i], mdz[:, i], den[:, i]
        subs[i] += 1
        s = np.clip(np.maximum(liq[:, i], 1e-6) / m / w, 0.01, 1.0)
        psi = -suc[:, i] * s ** -bb
        dpsi = -bb * psi / s / w
        nxt = lambda a: np.vstack([a[1:], a[-1:]])
        si = np.clip(np.where(bt, s, 0.5 * (s + nxt(s))), 0.01, 1.0)
        hk = hkc[:, i] * si ** (2.0 * bb + 3.0)
        dhk = (2.0 * bb + 3.0) * hk / si
        fall = nxt(psi) - psi
        d1, d2 = 0.5 * dhk / w, 0.5 * dhk / nxt(w)
        inner = lv & ~bt
        q = np.where(inner, hk - hk * fall / d, 0.0)
        q1 = np.where(inner, (hk * dpsi - d1 * fall) / d + d1, 0.0)
        q2 = np.where(inner, (-hk * nxt(dpsi) - d2 * fall) / d + d2, 0.0)
        up = lambda a, first: np.vstack([first, a[:-1]])
        zero = np.zeros((1, i.size))
        net = np.where(lv, up(q, c["qflx_infl"][None, i]) - q - sink[:, i], 0.0)
        r = dt[i] / m
        A = np.zeros((i.size, L, L))
        k = np.arange(L)
        A[:, k, k] = np.where(lv, -1.0 - (q1 - up(q2, zero)) * r, 1.0).T
        A[:, k[1:], k[:-1]] = np.where(lv, up(q1, zero) * r, 0.0)[1:].T
        A[:, k[:-1], k[1:]] = np.where(inner, -q2 * r, 0.0)[:-1].T
        x = np.linalg.solve(A, np.where(lv, -net * r, 0.0).T[..., None])[..., 0].T
        err = np.where(lv, np.abs(net - x / r) * dt[i] * 0.5, 0.0).max(axis=0)
        last = np.abs(DTIME - (done[i] + dt[i])) < 1e-8
        for name, a, rows in (("smp_l", psi, lv), ("hk_l", hk, lv), ("qin", up(q, c["qflx_infl"][None, i]), lv),
                              ("qout", q, lv)):
            sub = out[name][:L, i]
            out[name][:L, i] = np.where(rows & last, a, sub)
        again = (err > 0.1) & (dt[i] > 60.0)
        ok = i[~again]
        liq[:, ok] += np.where(lv, x * m, 0.0)[:, ~again]
        done[ok] += dt[ok]
        dt[i[again]] = np.maximum(dt[i[again]] / 2.0, 60.0)
        fin = np.abs(DTIME - done[ok]) < 1e-8
        grow = ok[(err[~again] < 0.01) & ~fin]
        dt[grow] *= 2.0
        dt[ok] = np.minimum(dt[ok], DTIME - done[ok])
        todo = np.concatenate([i[again], ok[~fin]])
        todo.sort()
    cap = c["eff_porosity"][:L] * mdz
    carry = np.zeros(n)
    for j in range(L - 1, -1, -1):
        wj = liq[j] + carry
        if j > 0:
            liq[j] = np.where(live[j], np.minimum(cap[j], wj), liq[j])
            carry = np.where(live[j], np.maximum(wj - cap[j], 0.0), carry)
        else:
            liq[j] = wj
    out["h2osoi_liq"][top] = np.where(live, liq, c["h2osoi_liq"][top])
    out["qcharge"], out["num_substeps"] = np.zeros(n), subs
    return out
