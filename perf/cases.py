"""What this framework is measured on: its hydro loop, through its public entry points.

A case is one segment of a user's program on state that the program already
holds on the GPU: a resident deck (`Chunk`), a batch of decks (`Ensemble`), a
program of the reference's own shape that calls the drop-in kernels one by one
on its host arrays (`clover_hip_*_kernel`), or the allocation-free summary of
device arrays.  The inputs are decks of the kind the repository runs
everywhere: a background state and a few cuboids or spheres of denser, hotter
gas in [0,10]^3, made from the seed.

What comes back is what such a program takes: the summary rows and the time
steps, and, where a field is small enough for a dump to be part of the segment,
the five fields of the state (density, energy and the three velocities).  The
largest meshes are run as the benchmark runs them, their fields staying on the
GPU and only the summaries and the step's dt reaching the host.
"""
import ctypes
import math
import random

import numpy as np
import torch

from cloverleaf3d_ref_amd import _lib
from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.deck import parse_deck
from cloverleaf3d_ref_amd.ensemble import Ensemble

STATE = ("density0", "energy0", "xvel0", "yvel0", "zvel0")

# "chunk": one deck.  form f64 | f32, tiles, states (2: one cuboid, 3: a
#   sphere too), steps per pass with a summary row every `every` steps, loop
#   run | step (clover_chunk_run, or a program that takes one step at a time
#   and reads its dt), tune (the launch-shape tuner runs once at set-up, as
#   bench.py and the clover.in program do), dump (the state's fields come back).
# "ensemble": `decks` decks of edges lo..hi in eights, advanced together.
# "dropin": the hydro loop of the reference over the drop-in kernels.
# "summary": field_summary of device arrays on a stream, without allocation.


def listed():
    return [
        # the reference's known-answer deck, one step at a time as the
        # clover.in program runs it: the smallest call, all latency
        dict(name="test_problem_10x2x2", kind="chunk", nx=10, ny=2, nz=2, form="f64", tiles=1, states=2, steps=75,
             every=75, loop="step", tune=False, dump=True),
        # the 64^3 cuboid deck that the tests and the CPU baseline run
        dict(name="cuboid_64", kind="chunk", nx=64, ny=64, nz=64, form="f64", tiles=1, states=2, steps=300, every=25,
             loop="run", tune=False, dump=True),
        # an odd, ragged mesh with three states
        dict(name="ragged_131x75x93", kind="chunk", nx=131, ny=75, nz=93, form="f64", tiles=1, states=3, steps=200,
             every=50, loop="run", tune=False, dump=True),
        # the FP32-store form on an odd mesh
        dict(name="ragged_f32_101x143x67", kind="chunk", nx=101, ny=143, nz=67, form="f32", tiles=1, states=3,
             steps=80, every=40, loop="run", tune=False, dump=False),
        # an ordinary mid-sized production mesh, launched with the defaults
        dict(name="cuboid_256", kind="chunk", nx=256, ny=256, nz=256, form="f64", tiles=1, states=2, steps=50, every=25,
             loop="run", tune=False, dump=False),
        # bench.py's headline workload in both forms
        dict(name="cuboid_512", kind="chunk", nx=512, ny=512, nz=512, form="f64", tiles=1, states=2, steps=25, every=25,
             loop="run", tune=True, dump=False),
        dict(name="cuboid_512_f32", kind="chunk", nx=512, ny=512, nz=512, form="f32", tiles=1, states=2, steps=25,
             every=25, loop="run", tune=True, dump=False),
        # bench.py's tiled workload at half its edge: internal halos
        dict(name="tiled_320_as_8", kind="chunk", nx=320, ny=320, nz=320, form="f64", tiles=8, states=2, steps=25,
             every=25, loop="run", tune=False, dump=False),
        # parameter studies: many small decks at once, in both forms
        dict(name="ensemble_48", kind="ensemble", decks=48, lo=16, hi=96, form="f64", steps=50, tune=True, dump=False),
        dict(name="ensemble_f32_24", kind="ensemble", decks=24, lo=16, hi=64, form="f32", steps=50, tune=False,
             dump=False),
        # a Fortran program that swapped its kernels for the drop-in ones
        dict(name="dropin_61x67x58", kind="dropin", nx=61, ny=67, nz=58, states=2, steps=100),
        # the summary inside somebody else's device program
        dict(name="summary_160x96x120", kind="summary", nx=160, ny=96, nz=120),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("chunk", "chunk", "chunk", "chunk", "ensemble", "dropin", "summary"))
    if kind == "ensemble":
        dump = rng.random() < 0.4
        decks = rng.randint(2, 6) if dump else _log_int(rng, 4, 64)
        hi = 8 * rng.randint(4, 6 if dump else 12)
        return dict(kind="ensemble", decks=decks, lo=8 * rng.randint(2, 3), hi=hi, form=rng.choice(("f64", "f32")),
                    steps=rng.choice((20, 50)), tune=rng.random() < 0.5, dump=dump)
    if kind == "dropin":
        return dict(kind="dropin", nx=_log_int(rng, 3, 70), ny=_log_int(rng, 3, 70), nz=_log_int(rng, 3, 70),
                    states=rng.choice((2, 3)), steps=rng.choice((50, 100)))
    if kind == "summary":
        return dict(kind="summary", nx=_log_int(rng, 8, 200), ny=_log_int(rng, 8, 200), nz=_log_int(rng, 8, 200))
    dump = rng.random() < 0.5
    lo, hi = (2, 100) if dump else (60, 400)
    nx, ny, nz = (_log_int(rng, lo, hi) for _ in range(3))
    cells = nx * ny * nz
    tiles = rng.choice((2, 4, 8)) if min(nx, ny, nz) >= 16 and rng.random() < 0.25 else 1
    form = rng.choice(("f64", "f64", "f32"))
    # an FP32 run is a run of its own after some hundred steps: shorter ones can be compared
    steps = (40 if form == "f32" else 200) if dump else max(10, min(60, int(1.5e9 / cells) // 10 * 10))
    return dict(kind="chunk", nx=nx, ny=ny, nz=nz, form=form, tiles=tiles,
                states=rng.choice((2, 3)), steps=steps, every=steps if rng.random() < 0.5 else steps // 2,
                loop=rng.choice(("run", "run", "step")), tune=not dump and rng.random() < 0.4, dump=dump)


# ---------------------------------------------------------------- the inputs
def _states(rng, states):
    """The background and `states`-1 regions: cuboids, then a sphere."""
    out = [dict(density=rng.uniform(0.1, 0.5), energy=rng.uniform(0.5, 1.5))]
    for s in range(1, states):
        st = dict(density=rng.uniform(0.5, 2.0), energy=rng.uniform(1.5, 5.0))
        if s == 2:
            st.update(geometry="sphere", radius=rng.uniform(1.0, 2.5))
            for a in "xyz":
                st[a + "min"] = rng.uniform(3.0, 7.0)  # the centre
        else:
            st["geometry"] = "cuboid"
            for a in "xyz":
                length = rng.uniform(1.0, 4.0)
                st[a + "min"] = rng.uniform(0.0, 10.0 - length)
                st[a + "max"] = st[a + "min"] + length
        out.append(st)
    return out


def _deck_text(n, states, every, tiles=1):
    lines = ["*clover"]
    for i, st in enumerate(states, 1):
        lines.append(" state %d " % i + " ".join("%s=%s" % (k, v if isinstance(v, str) else repr(v))
                                                for k, v in st.items()))
    lines += [" %s_cells=%d" % (a, c) for a, c in zip("xyz", n)]
    lines += [" %smin=0.0\n %smax=10.0" % (a, a) for a in "xyz"]
    lines += [" initial_timestep=0.04", " timestep_rise=1.5", " end_time=1.0e9", " end_step=2000000000",
              " summary_frequency=%d" % every, " tiles_per_chunk %d" % tiles]
    if tiles > 1:
        lines.append(" 3d_tile_decomposition")
    return "\n".join(lines + ["*endclover", ""])


def _ensemble_sizes(case):
    """The decks' meshes, the same for every seed."""
    rng = random.Random(case["decks"] * 1000 + case["hi"])
    edges = range(case["lo"], case["hi"] + 1, 8)
    return [tuple(rng.choice(edges) for _ in range(3)) for _ in range(case["decks"])]


def _ensemble_inputs(case, seed):
    rng = random.Random(seed)
    return [(n, _states(rng, 2)) for n in _ensemble_sizes(case)]


def _sizes(case):
    return case["nx"], case["ny"], case["nz"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "chunk":
        states = _states(random.Random(seed), case["states"])
        deck = parse_deck(_deck_text(_sizes(case), states, case["every"], case["tiles"]))
        chunk = Chunk(deck, fp32=case["form"] == "f32")
        if case["tune"]:
            chunk.autotune()
        return dict(case, chunk=chunk)
    if kind == "ensemble":
        decks = [parse_deck(_deck_text(n, states, 0)) for n, states in _ensemble_inputs(case, seed)]
        ens = Ensemble(decks, fp32=case["form"] == "f32")
        if case["tune"]:
            ens.autotune()
        return dict(case, ensemble=ens, decks=decks)
    if kind == "dropin":
        return dict(case, program=DropIn(_sizes(case), _states(random.Random(seed), case["states"])))
    return dict(case, summary=DeviceSummary(_summary_arrays(case, seed)))


def _interior(a, nodes):
    """The computed cells or nodes of a fetched field; its halo holds whatever the last exchange left."""
    e = 3 if nodes else 2
    return a[tuple(slice(2, s - e + (1 if nodes else 0)) for s in a.shape)]


def _field(a, name, form):
    a = _interior(a, name[1:4] == "vel")
    return a.astype(np.float32) if form == "f32" else a


def _numbers(v, form):
    """Totals and times, at the precision their form has."""
    return np.array(v, dtype=np.float32 if form == "f32" else np.float64)


def run(state):
    kind = state["kind"]
    if kind == "chunk":
        c, out = state["chunk"], {}
        if state["loop"] == "step":
            dts = [c.step() for _ in range(state["steps"])]
            rows = [c.field_summary()]
        else:
            rows = c.run(state["steps"])
            dts = [c.state()[2]]
        out["dt"] = _numbers(dts, state["form"])
        out["rows"] = _numbers([[r[k] for k in ROW] for r in rows], state["form"])
        if state["dump"]:
            out["tiles"] = [[_field(c.fetch(f, t), f, state["form"]) for f in STATE] for t in range(c.ntiles)]
        return out
    if kind == "ensemble":
        e = state["ensemble"]
        e.run(state["steps"])
        rows = [[s[k] for k in SUMS] for s in e.summaries()]
        _, time, dt, _ = e.state()
        out = {k: _numbers(v, state["form"]) for k, v in (("rows", rows), ("time", time), ("dt", dt))}
        if state["dump"]:
            out["decks"] = [[_field(e.fetch(d, f), f, state["form"]) for f in STATE]
                            for d in range(len(state["decks"]))]
        return out
    if kind == "dropin":
        return state["program"].run(state["steps"])
    return state["summary"].run()


SUMS = ("vol", "mass", "ie", "ke", "press")
ROW = ("time",) + SUMS


# ------------------------------------------------------ the drop-in program
HALO = (("density0", "C"), ("energy0", "C"), ("pressure", "C"), ("viscosity", "C"), ("soundspeed", "C"),
        ("density1", "C"), ("energy1", "C"), ("xvel0", "V"), ("yvel0", "V"), ("zvel0", "V"), ("xvel1", "V"),
        ("yvel1", "V"), ("zvel1", "V"), ("vol_flux_x", "X"), ("vol_flux_y", "Y"), ("vol_flux_z", "Z"),
        ("mass_flux_x", "X"), ("mass_flux_y", "Y"), ("mass_flux_z", "Z"))
FLAGS = ("density0", "density1", "energy0", "energy1", "pressure", "viscosity", "soundspeed", "xvel0", "xvel1",
         "yvel0", "yvel1", "zvel0", "zvel1", "vol_flux_x", "vol_flux_y", "vol_flux_z", "mass_flux_x", "mass_flux_y",
         "mass_flux_z")  # the order of the reference's field flags
CLASS = dict(HALO, volume="C", xarea="X", yarea="Y", zarea="Z", **{"work%d" % i: "V" for i in range(1, 8)})
SAFE = dict(dtc=0.75, dtu=0.5, dtv=0.5, dtw=0.5, dtdiv=0.5)
G_SMALL, G_BIG = float(np.float32(1.0e-16)), float(np.float32(1.0e21))


def _shape(cls, n):
    return tuple(c + 4 + (cls == "V" or cls == a) for c, a in zip(n, "XYZ"))


class DropIn:
    """A program with the reference's arrays and call order that calls the
    drop-in kernels: its arrays are host arrays in Fortran order, which stay on
    the GPU from the first call that sees them until the program fetches them."""

    def __init__(self, n, states):
        self.n, self.L = n, _lib.lib()
        _lib.check(self.L.clover_hip_init(0), "clover_hip_init")
        a = self.a = {k: np.zeros(_shape(cls, n), order="F") for k, cls in CLASS.items()}
        d = [10.0 / c for c in n]
        for ax, c, h in zip("xyz", n, d):
            vertex = h * np.arange(-2, c + 3)
            a["cell" + ax] = 0.5 * (vertex[1:] + vertex[:-1])
            a["celld" + ax], a["vertexd" + ax] = np.full(c + 4, h), np.full(c + 5, h)
        a["volume"][:], a["xarea"][:] = d[0] * d[1] * d[2], d[1] * d[2]
        a["yarea"][:], a["zarea"][:] = d[0] * d[2], d[0] * d[1]
        rho, e = _paint(n, states)
        a["density0"][:], a["energy0"][:] = rho.T, e.T
        self.p = {k: ctypes.c_void_p(v.ctypes.data) for k, v in a.items()}
        self.dims = [x for c in n for x in (1, c)]
        self.out_d, self.out_i = (ctypes.c_double * 5)(), (ctypes.c_int * 5)()
        self.external = (ctypes.c_int * 6)(*[-1] * 6)
        self.dtold, self.time, self.advect_x = 0.04, 0.0, 1
        # the argument lists that do not change from step to step
        self.halos = {k: self._halo_args(fields, depth) for k, (fields, depth) in EXCHANGES.items()}
        self._call("ideal_gas", self._args("density0 energy0 pressure soundspeed"))
        self._halo("start")

    def __del__(self):
        for p in getattr(self, "p", {}).values():
            self.L.clover_hip_forget(p)

    def _args(self, names):
        return [self.p[k] for k in names.split()]

    def _call(self, kernel, args):
        if getattr(self.L, "clover_hip_%s_kernel" % kernel)(*self.dims, *args):
            raise RuntimeError(self.L.clover_hip_last_error().decode())

    def _halo_args(self, fields, depth):
        flags = (ctypes.c_int * 19)(*[int(f in fields.split()) for f in FLAGS])
        return [self.external, self.external] + [self.p[k] for k, _ in HALO] + [flags, depth]

    def _halo(self, which):
        self._call("update_halo", self.halos[which])

    def _pdv(self, predict, dt):
        args = self._args("xarea yarea zarea volume density0 density1 energy0 energy1 pressure viscosity xvel0 xvel1"
                          " yvel0 yvel1 zvel0 zvel1")
        if self.L.clover_hip_PdV_kernel(predict, *self.dims, ctypes.c_double(dt), *args):
            raise RuntimeError(self.L.clover_hip_last_error().decode())

    def _advec_cell(self, sweep, direction):
        self._call("advec_cell", [self.advect_x, direction, sweep] + self._args(
            "vertexdx vertexdy vertexdz volume density1 energy1 mass_flux_x vol_flux_x mass_flux_y vol_flux_y"
            " mass_flux_z vol_flux_z work1 work2 work3 work4 work5 work6 work7"))

    def _advec_mom(self, sweep, direction):
        rest = self._args("mass_flux_x vol_flux_x mass_flux_y vol_flux_y mass_flux_z vol_flux_z volume density1 work1"
                          " work2 work3 work4 work5 work6 work7 celldx celldy celldz")
        for which, vel in enumerate(("xvel1", "yvel1", "zvel1"), 1):
            self._call("advec_mom", [self.p[vel]] + rest + [self.advect_x, which, sweep, direction])

    def _timestep(self):
        self._call("ideal_gas", self._args("density0 energy0 pressure soundspeed"))
        self._halo("timestep")
        self._call("viscosity", self._args("xarea yarea zarea celldx celldy celldz density0 pressure viscosity xvel0"
                                           " yvel0 zvel0"))
        self._halo("viscosity")
        d, i = self.out_d, self.out_i
        at = [ctypes.byref(d, 8 * q) for q in range(5)]
        ai = [ctypes.byref(i, 4 * q) for q in range(5)]
        c = ctypes.c_double
        self._call("calc_dt", [c(G_SMALL), c(G_BIG), c(1.0e-7)] + [c(SAFE[k]) for k in SAFE] + self._args(
            "xarea yarea zarea cellx celly cellz celldx celldy celldz volume density0 energy0 pressure viscosity"
            " soundspeed xvel0 yvel0 zvel0 work1") + [at[0], ai[0], at[1], at[2], at[3], ai[1], ai[2], ai[3], ai[4]])
        self.dtold = min(min(G_BIG, d[0]), self.dtold * 1.5, 1.0)
        return self.dtold

    def _step(self):
        dt = self._timestep()
        c = ctypes.c_double(dt)
        self._pdv(1, dt)
        self._call("ideal_gas", self._args("density1 energy1 pressure soundspeed"))
        self._halo("pressure")
        self._call("revert", self._args("density0 density1 energy0 energy1"))
        self._call("accelerate", [c] + self._args("xarea yarea zarea volume density0 pressure viscosity xvel0 yvel0"
                                                  " zvel0 xvel1 yvel1 zvel1"))
        self._pdv(0, dt)
        self._call("flux_calc", [c] + self._args("xarea yarea zarea xvel0 yvel0 zvel0 xvel1 yvel1 zvel1 vol_flux_x"
                                                 " vol_flux_y vol_flux_z"))
        first, last = (1, 3) if self.advect_x else (3, 1)
        for sweep, direction in ((1, first), (2, 2), (3, last)):
            if sweep < 3:
                self._halo("cells")
            self._advec_cell(sweep, direction)
            self._halo("momentum")
            self._advec_mom(sweep, direction)
        self._call("reset_field", self._args("density0 density1 energy0 energy1 xvel0 xvel1 yvel0 yvel1 zvel0 zvel1"))
        self.advect_x = 1 - self.advect_x
        self.time += dt
        return dt

    def run(self, steps):
        dts = np.array([self._step() for _ in range(steps)])
        self._call("ideal_gas", self._args("density0 energy0 pressure soundspeed"))
        at = [ctypes.byref(self.out_d, 8 * q) for q in range(5)]
        self._call("field_summary", self._args("volume density0 energy0 pressure xvel0 yvel0 zvel0") + at)
        rows = np.array([[self.time] + list(self.out_d)])
        for f in STATE:
            _lib.check(self.L.clover_hip_fetch(self.p[f]), "clover_hip_fetch")
        return dict(dt=dts, rows=rows, tiles=[[_interior(self.a[f], f[1:4] == "vel") for f in STATE]])


# the reference's exchanges: the fields each flags, and its depth
EXCHANGES = {
    "start": ("density0 energy0 pressure viscosity density1 energy1 xvel0 yvel0 zvel0 xvel1 yvel1 zvel1", 2),
    "timestep": ("pressure energy0 density0 xvel0 yvel0", 1),
    "viscosity": ("viscosity", 1),
    "pressure": ("pressure", 1),
    "cells": ("energy1 density1 vol_flux_x vol_flux_y vol_flux_z", 2),
    "momentum": ("density1 energy1 xvel1 yvel1 zvel1 mass_flux_x mass_flux_y mass_flux_z", 2),
}


# ------------------------------------------------- the allocation-free summary
def _summary_arrays(case, seed):
    """volume, density0, energy0, pressure, xvel0, yvel0, zvel0 in the reference's shapes (x fastest)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    cell, node = (tuple(reversed(_shape(c, _sizes(case)))) for c in "CV")

    def uniform(shape, lo, hi):
        return torch.rand(shape, dtype=torch.float64, device="cuda", generator=g) * (hi - lo) + lo

    nx, ny, nz = _sizes(case)
    volume = torch.full(cell, 1000.0 / (nx * ny * nz), dtype=torch.float64, device="cuda")
    rho, e = uniform(cell, 0.1, 2.0), uniform(cell, 0.5, 5.0)
    return [volume, rho, e, 0.4 * rho * e] + [uniform(node, -1.0, 1.0) for _ in range(3)], _sizes(case)


class DeviceSummary:
    def __init__(self, made):
        self.arrays, n = made
        self.sums = torch.zeros(5, dtype=torch.float64, device="cuda")
        self.fn = _lib.lib().clover_hip_field_summary_kernel_noalloc
        self.args = [x for c in n for x in (1, c)] + [ctypes.c_void_p(t.data_ptr()) for t in self.arrays + [self.sums]]

    def run(self):
        if self.fn(*self.args, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)):
            raise RuntimeError("clover_hip_field_summary_kernel_noalloc failed")
        return self.sums


# ----------------------------------------------------------------------- work
FLOPS_PER_CELL_STEP = 850  # additions, products, quotients and roots of the reference's loop nests


def _cells(case):
    if case["kind"] == "ensemble":
        return sum(nx * ny * nz for nx, ny, nz in _ensemble_sizes(case))
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    cells = _cells(case)
    if case["kind"] == "summary":
        return dict(bytes=56.0 * cells, flops=66.0 * cells)
    # a step reads the state's five fields and writes their new values
    size = 4 if case.get("form") == "f32" else 8
    b = 10.0 * size * cells * case["steps"]
    if case.get("dump", case["kind"] == "dropin"):
        b += 5.0 * size * cells
    return dict(bytes=b, flops=float(FLOPS_PER_CELL_STEP) * cells * case["steps"])


# ---------------------------------------------------------------------- exact
# The reference's step in 64 bits on whole arrays.  An array is (z, y, x) with
# index 0 = min-2; every class has the vertex extents.  R(j0, j1, k0, k1, l0,
# l1) is a range of the reference's indices, both ends included.
def _paint(n, states):
    """density0 and energy0 of every cell, halo included, as (z, y, x) arrays."""
    d = [10.0 / c for c in n]
    low = [h * np.arange(-2, c + 2) for c, h in zip(n, d)]
    high = [h * np.arange(-1, c + 3) for c, h in zip(n, d)]
    mid = [0.5 * (a + b) for a, b in zip(low, high)]
    shape = tuple(reversed([c + 4 for c in n]))
    rho, e = np.full(shape, states[0]["density"]), np.full(shape, states[0]["energy"])
    for st in states[1:]:
        lo = [st[a + "min"] + h / 100.0 for a, h in zip("xyz", d)]
        if st["geometry"] == "sphere":
            r2 = [(m - c) * (m - c) for m, c in zip(mid, lo)]
            hit = np.sqrt(r2[0][None, None, :] + r2[1][None, :, None] + r2[2][:, None, None]) <= st["radius"]
        else:
            hi = [st[a + "max"] - h / 100.0 for a, h in zip("xyz", d)]
            x, y, z = ((b >= q) & (a < r) for a, b, q, r in zip(low, high, lo, hi))
            hit = x[None, None, :] & y[None, :, None] & z[:, None, None]
        rho[hit], e[hit] = st["density"], st["energy"]
    return rho, e


# per field: how it sits on each axis (0 cell, 1 staggered, 2 face data
# tangential to the axis), the axis along which it flips sign, and, per face,
# what the face's two tangential ranges reach beyond max+depth
_CELLS = ("density0", "density1", "energy0", "energy1", "pressure", "viscosity", "soundspeed")
_SIT = {**{f: (0, 0, 0) for f in _CELLS}, **{a + "vel" + i: (1, 1, 1) for a in "xyz" for i in "01"},
        **{q + "_flux_x": (1, 2, 2) for q in ("vol", "mass")}, **{q + "_flux_y": (2, 1, 2) for q in ("vol", "mass")},
        **{q + "_flux_z": (2, 2, 1) for q in ("vol", "mass")}}


def _normal(f):
    return "xyz".index(f[0]) if f[1:4] == "vel" else "xyz".index(f[-1]) if "flux" in f else -1


def _beyond(f, axis, high):
    if f[1:4] == "vel":
        return 1, 1
    if "flux" not in f or f[-1] == "xyz"[axis]:
        return 0, 0
    tangential = [a for a in range(3) if a != axis]
    ext = [int(f[-1] == "xyz"[a]) for a in tangential]
    if f == "vol_flux_z" and axis == 1 and not high:
        ext = [0, 0]
    if f[-1] in "xy" and axis == 2:
        ext = [0, 0]
    return tuple(ext)


class Exact:
    def __init__(self, n, states, device):
        self.n = n
        self.f = {k: torch.zeros(tuple(c + 5 for c in reversed(n)), dtype=torch.float64, device=device) for k in _SIT}
        rho, e = _paint(n, states)
        for name, v in (("density0", rho), ("energy0", e)):
            self.f[name][:-1, :-1, :-1] = torch.from_numpy(v).to(device)
        self.d = [10.0 / c for c in n]
        self.vol = self.d[0] * self.d[1] * self.d[2]
        self.area = (self.d[1] * self.d[2], self.d[0] * self.d[2], self.d[0] * self.d[1])
        self.dt = self.dtold = 0.04
        self.time, self.advect_x = 0.0, True
        self.cells = self.R(1, n[0], 1, n[1], 1, n[2])
        self.nodes = self.R(1, n[0] + 1, 1, n[1] + 1, 1, n[2] + 1)
        self.ideal_gas("0")
        self.halo("start")

    @staticmethod
    def R(*r):
        return r

    def at(self, a, r, j=0, k=0, l=0):  # noqa: E741
        a = self.f[a] if isinstance(a, str) else a
        return a[r[4] + 1 + l:r[5] + 2 + l, r[2] + 1 + k:r[3] + 2 + k, r[0] + 1 + j:r[1] + 2 + j]

    def put(self, a, r, v):
        self.at(a, r).copy_(v)

    def along(self, a, r, axis, q):
        return self.at(a, r, *[q if x == axis else 0 for x in range(3)])

    def halo(self, which):
        fields, depth = EXCHANGES[which]
        for f in fields.split():
            for axis in (1, 0, 2):
                m, sit = self.n[axis], _SIT[f][axis]
                sign = -1.0 if _normal(f) == axis else 1.0
                tangential = [a for a in range(3) if a != axis]
                for high in (0, 1):
                    ext = _beyond(f, axis, high)
                    for d in range(1, depth + 1):
                        if not high:
                            w, r = 1 - d, d if sit == 0 else 1 + d
                        elif sit == 0:
                            w, r = m + d, m + 1 - d
                        elif sit == 1:
                            w, r = m + 1 + d, m + 1 - d
                        else:
                            w, r = m + d, m - d
                        sl = [None] * 3
                        for a, x in zip(tangential, ext):
                            sl[a] = slice(2 - depth, self.n[a] + depth + x + 2)
                        src, dst = list(sl), list(sl)
                        src[axis], dst[axis] = r + 1, w + 1
                        self.f[f][tuple(reversed(dst))] = sign * self.f[f][tuple(reversed(src))]

    def ideal_gas(self, level):
        rho, e = self.at("density" + level, self.cells), self.at("energy" + level, self.cells)
        v = 1.0 / rho
        p = (1.4 - 1.0) * rho * e
        self.put("pressure", self.cells, p)
        self.put("soundspeed", self.cells, torch.sqrt(v * v * (p * (1.4 - 1.0) * rho + rho * p)))

    def corners(self, name, r, axis, side):
        """The sum of the four nodes of the cell's low (0) or high (1) face along `axis`."""
        other = [a for a in range(3) if a != axis]
        s = 0.0
        for b in (0, 1):
            for a in (0, 1):
                q = [0, 0, 0]
                q[axis], q[other[0]], q[other[1]] = side, a, b
                s = s + self.at(name, r, *q)
        return s

    def viscosity(self):
        r, d = self.cells, self.d
        grad = [[self.corners(v, r, ax, 1) - self.corners(v, r, ax, 0) for ax in range(3)]
                for v in ("xvel0", "yvel0", "zvel0")]
        div = (self.area[0] * grad[0][0] + self.area[1] * grad[1][1]) + self.area[2] * grad[2][2]
        xx, yy, zz = (0.25 * grad[a][a] / d[a] for a in range(3))
        xy = 0.25 * grad[0][1] / d[1] + 0.25 * grad[1][0] / d[0]
        xz = 0.25 * grad[0][2] / d[2] + 0.25 * grad[2][0] / d[0]
        yz = 0.25 * grad[1][2] / d[2] + 0.25 * grad[2][1] / d[1]
        del grad
        pg = [(self.along("pressure", r, a, 1) - self.along("pressure", r, a, -1)) / (2.0 * d[a]) for a in range(3)]
        x2, y2, z2 = (p * p for p in pg)
        limiter = (xx * x2 + yy * y2 + zz * z2 + xy * pg[0] * pg[1] + xz * pg[0] * pg[2] + yz * pg[1] * pg[2]) / \
            (x2 + y2 + z2).clamp_min(1.0e-16)
        pg = [torch.copysign(p.abs().clamp_min(1.0e-16), p) for p in pg]
        pgrad = torch.sqrt(pg[0] * pg[0] + pg[1] * pg[1] + pg[2] * pg[2])
        g = [(d[a] * pgrad / pg[a]).abs() for a in range(3)]
        g = torch.minimum(torch.minimum(g[0], g[1]), g[2])
        q = 2.0 * self.at("density0", r) * g * g * limiter * limiter
        self.put("viscosity", r, torch.where((limiter > 0.0) | (div >= 0.0), torch.zeros_like(q), q))

    def calc_dt(self):
        r, h = self.cells, min(self.d)
        c = self.at("soundspeed", r)
        cc = c * c + 2.0 * self.at("viscosity", r) / self.at("density0", r)
        dt = (SAFE["dtc"] / torch.sqrt(cc / (h * h)).clamp_min(G_SMALL)).amin()
        div = 0.0
        for a, (v, s) in enumerate((("xvel0", "dtu"), ("yvel0", "dtv"), ("zvel0", "dtw"))):
            lo, hi = (self.corners(v, r, a, side) * self.area[a] for side in (0, 1))
            big = torch.maximum(lo.abs(), hi.abs()).clamp_min(1.0e-5 * self.vol).amax()
            dt = torch.minimum(dt, SAFE[s] * 4.0 * self.vol / big)
            div = div + hi - lo
        dt = torch.minimum(dt, SAFE["dtdiv"] * 4.0 * self.vol / div.abs().clamp_min(self.vol * 1.0e-5).amax())
        self.dt = self.dtold = min(float(dt), G_BIG, self.dtold * 1.5, 1.0)

    def pdv(self, dt, other):
        r = self.cells
        total = 0.0
        for a, v in enumerate("xyz"):
            for side, sign in ((1, 1.0), (0, -1.0)):
                s = self.corners(v + "vel0", r, a, side) + self.corners(v + "vel" + other, r, a, side)
                total = total + sign * (self.area[a] * s * 0.125 * dt)
        rho = self.at("density0", r)
        change = (self.at("pressure", r) / rho + self.at("viscosity", r) / rho) * total / self.vol
        self.put("energy1", r, self.at("energy0", r) - change)
        self.put("density1", r, rho * (self.vol / (self.vol + total)))

    def accelerate(self):
        r = self.nodes
        eight = [(a, b, c) for c in (0, -1) for b in (-1, 0) for a in (-1, 0)]
        step = 0.25 * self.dt / (0.125 * self.vol * sum(self.at("density0", r, *q) for q in eight))
        for ax, v in enumerate("xyz"):
            new = self.at(v + "vel0", r)
            for name in ("pressure", "viscosity"):
                s = 0.0
                for q in eight:
                    s = s + (1.0 if q[ax] == 0 else -1.0) * self.at(name, r, *q)
                new = new - step * (self.area[ax] * s)
            self.put(v + "vel1", r, new)

    def flux_calc(self):
        n = self.n
        for ax, v in enumerate("xyz"):
            r = [1, n[0], 1, n[1], 1, n[2]]
            r[2 * ax + 1] += 1
            if v == "z":  # the reference adds zvel0(j+1,k,l) twice and zvel0(j,k+1,l) not at all
                s = self.corners("zvel1", r, 2, 0) + self.at("zvel0", r) + 2.0 * self.at("zvel0", r, 1) + \
                    self.at("zvel0", r, 1, 1)
            else:
                s = self.corners(v + "vel0", r, ax, 0) + self.corners(v + "vel1", r, ax, 0)
            self.put("vol_flux_" + v, r, 0.125 * self.dt * self.area[ax] * s)

    def volume_change(self, r, axes):
        s = 0.0
        for a in axes:
            f = "vol_flux_" + "xyz"[a]
            s = s + (self.along(f, r, a, 1) - self.at(f, r))
        return s

    def limited(self, sigma, upwind, donor, downwind):
        up, down = donor - upwind, downwind - donor
        low = torch.minimum(torch.minimum(up.abs(), down.abs()),
                            ((1.0 + sigma) * up.abs() + (2.0 - sigma) * down.abs()) / 6.0)
        return torch.where(up * down > 0.0, (1.0 - sigma) * torch.copysign(low, down), torch.zeros_like(low))

    def advec_cell(self, sweep, ax):
        n, order = self.n, (0, 1, 2) if self.advect_x else (2, 1, 0)
        every = self.R(-1, n[0] + 2, -1, n[1] + 2, -1, n[2] + 2)
        pre = torch.zeros_like(self.f["density1"])
        self.put(pre, every, self.vol + self.volume_change(every, order[sweep - 1:]))
        r = [1, n[0], 1, n[1], 1, n[2]]
        r[2 * ax + 1] += 2
        if ax == 1:
            r[5] += 2  # the y sweep's faces run two planes past z_max
        vf = self.at("vol_flux_" + "xyz"[ax], r)
        up = vf > 0.0

        def sides(name):
            """upwind, donor and downwind cells of each face; the upwind one of the last face stays inside the halo"""
            a = self.f[name] if isinstance(name, str) else name
            beyond = self.along(a, r, ax, 0).clone()
            cut = [slice(None)] * 3
            cut[2 - ax] = slice(0, -1)
            src = list(cut)
            src[2 - ax] = slice(1, None)
            beyond[tuple(cut)] = self.along(a, r, ax, 0)[tuple(src)]
            lo2, lo1, here = (self.along(a, r, ax, q) for q in (-2, -1, 0))
            return torch.where(up, lo2, beyond), torch.where(up, lo1, here), torch.where(up, here, lo1)

        donor_vol = torch.where(up, self.along(pre, r, ax, -1), self.at(pre, r))
        sigma = vf.abs() / donor_vol
        u, c, w = sides("density1")
        mass = vf * (c + self.limited(sigma, u, c, w))
        sigma_m = mass.abs() / (c * donor_vol)
        u, c, w = sides("energy1")
        ener = torch.zeros_like(pre)
        lim = self.limit_energy(sigma_m, sigma, u, c, w)
        self.put(ener, r, mass * (c + lim))
        self.put("mass_flux_" + "xyz"[ax], r, mass)
        r = self.cells
        mf, pv = self.f["mass_flux_" + "xyz"[ax]], self.at(pre, r)
        pm = self.at("density1", r) * pv
        pom = pm + self.at(mf, r) - self.along(mf, r, ax, 1)
        e = (self.at("energy1", r) * pm + self.at(ener, r) - self.along(ener, r, ax, 1)) / pom
        f = "vol_flux_" + "xyz"[ax]
        rho = pom / (pv + self.at(f, r) - self.along(f, r, ax, 1))
        self.put("energy1", r, e)
        self.put("density1", r, rho)

    def limit_energy(self, sigma_m, sigma, upwind, donor, downwind):
        up, down = donor - upwind, downwind - donor
        low = torch.minimum(torch.minimum(up.abs(), down.abs()),
                            ((1.0 + sigma) * up.abs() + (2.0 - sigma) * down.abs()) / 6.0)
        return torch.where(up * down > 0.0, (1.0 - sigma_m) * torch.copysign(low, down), torch.zeros_like(low))

    def advec_mom(self, sweep, ax):
        n, order = self.n, (0, 1, 2) if self.advect_x else (2, 1, 0)
        every = self.R(-1, n[0] + 2, -1, n[1] + 2, -1, n[2] + 2)
        mass = torch.zeros_like(self.f["density1"])
        self.put(mass, every, self.at("density1", every) * (self.vol + self.volume_change(every, order[sweep:])))
        other = [a for a in range(3) if a != ax]

        def span(lo, hi):
            r = [1, n[0] + 1, 1, n[1] + 1, 1, n[2] + 1]
            r[2 * ax], r[2 * ax + 1] = lo, n[ax] + hi
            return r

        def near(a, r, along):
            s = 0.0
            for p in along:
                for b in (0, -1):
                    for c in (0, -1):
                        q = [0, 0, 0]
                        q[ax], q[other[0]], q[other[1]] = p, b, c
                        s = s + self.at(a, r, *q)
            return 0.125 * s

        nf, pre, post, flux = (torch.zeros_like(mass) for _ in range(4))
        r = span(-1, 2)
        self.put(nf, r, near("mass_flux_" + "xyz"[ax], r, (0, 1)))
        r = span(0, 2)
        self.put(post, r, near(mass, r, (0, -1)))
        self.put(pre, r, self.at(post, r) - self.along(nf, r, ax, -1) + self.at(nf, r))
        faces = span(0, 1)
        f = self.at(nf, faces)
        back = f < 0.0
        sigma = f.abs() / torch.where(back, self.along(pre, faces, ax, 1), self.at(pre, faces))
        for v in ("xvel1", "yvel1", "zvel1"):
            m1, c0, p1, p2 = (self.along(v, faces, ax, q) for q in (-1, 0, 1, 2))
            donor = torch.where(back, p1, c0)
            lim = self.limited(sigma, torch.where(back, p2, m1), donor, torch.where(back, c0, p1))
            self.put(flux, faces, (donor + lim) * f)
            r = self.nodes
            self.put(v, r, (self.at(v, r) * self.at(pre, r) + self.along(flux, r, ax, -1) - self.at(flux, r)) /
                     self.at(post, r))

    def step(self):
        self.ideal_gas("0")
        self.halo("timestep")
        self.viscosity()
        self.halo("viscosity")
        self.calc_dt()
        self.pdv(0.5 * self.dt, "0")
        self.ideal_gas("1")
        self.halo("pressure")
        self.accelerate()
        self.pdv(self.dt, "1")
        self.flux_calc()
        order = (0, 1, 2) if self.advect_x else (2, 1, 0)
        for sweep, ax in enumerate(order, 1):
            if sweep < 3:
                self.halo("cells")
            self.advec_cell(sweep, ax)
            self.halo("momentum")
            self.advec_mom(sweep, ax)
        for name in ("density", "energy"):
            self.put(name + "0", self.cells, self.at(name + "1", self.cells))
        for name in ("xvel", "yvel", "zvel"):
            self.put(name + "0", self.nodes, self.at(name + "1", self.nodes))
        self.advect_x = not self.advect_x
        self.time += self.dt
        return self.dt

    def sums(self):
        self.ideal_gas("0")
        r = self.cells
        rho, e, p = (self.at(f, r) for f in ("density0", "energy0", "pressure"))
        v2 = 0.0
        for v in ("xvel0", "yvel0", "zvel0"):
            for q in range(8):
                x = self.at(v, r, q & 1, q >> 1 & 1, q >> 2)
                v2 = v2 + 0.125 * (x * x)
        mass = self.vol * rho
        return [self.vol * rho.numel()] + [float(t.sum()) for t in (mass, mass * e, mass * 0.5 * v2, self.vol * p)]

    def field(self, name):
        """As the program holds it: x first."""
        return self.at(name, self.nodes if name[1:4] == "vel" else self.cells).permute(2, 1, 0).cpu().numpy().copy()

    def state(self):
        """The state's fields; None for a velocity that only rounding keeps from zero (a symmetric thin mesh)."""
        fields = [self.field(f) for f in STATE]
        return [None if np.abs(a).max() < 1.0e-10 else a for a in fields]


def exact(case, seed):
    kind = case["kind"]
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "summary":
        (volume, rho, e, p, *vel), n = _summary_arrays(case, seed)
        inner = tuple(slice(2, 2 + c) for c in reversed(n))
        v2 = 0.0
        for v in vel:
            for q in range(8):
                x = v[tuple(slice(s.start + (q >> b & 1), s.stop + (q >> b & 1)) for s, b in zip(inner, (2, 1, 0)))]
                v2 = v2 + 0.125 * (x * x)
        volume, rho, e, p = (t[inner] for t in (volume, rho, e, p))
        return torch.stack([t.sum() for t in (volume, volume * rho, volume * rho * e, volume * rho * 0.5 * v2,
                                              volume * p)])
    if kind == "ensemble":
        if case["decks"] * case["steps"] > 1200:
            return None  # one deck after another: minutes
        rows, times, dts, fields = [], [], [], []
        for n, states in _ensemble_inputs(case, seed):
            x = Exact(n, states, device)
            for _ in range(case["steps"]):
                x.step()
            rows.append(x.sums())
            times.append(x.time)
            dts.append(x.dt)
            fields.append(x.state() if case["dump"] else None)
        out = dict(rows=np.array(rows), time=np.array(times), dt=np.array(dts))
        return dict(out, decks=fields) if case["dump"] else out
    steps = case["steps"]
    if _cells(case) * steps > 4.0e9 or case.get("tiles", 1) > 1:
        return None  # too long; and the reference's exchanges between tiles change values at the 1e-6 level
    x = Exact(_sizes(case), _states(random.Random(seed), case["states"]), device)
    every = case.get("every", steps)
    stepping = kind == "dropin" or case["loop"] == "step"
    dts, rows = [], []
    for s in range(1, steps + 1):
        dts.append(x.step())
        if s == steps if stepping else s % every == 0:
            rows.append([x.time] + x.sums())
    out = dict(dt=np.array(dts if stepping else dts[-1:]), rows=np.array(rows))
    if case.get("dump", kind == "dropin"):
        out["tiles"] = [x.state()]
    return out

