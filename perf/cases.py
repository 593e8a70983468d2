"""Performance cases of the FDTD engine: what programs written against include/alis.h have it do.

Every case but two builds its worlds with the public C API through ctypes (createWorld,
putObjectArray, pointDipole, planewave, createPhasers) and one pass is the body of such a program:
a run of time steps with its per-step reads, then what the program takes home -- the fields
(syncWorld, as timer() does at the end of a loop), the net flux of its phasers, its probe values.
The far-field case is the evaluation that follows a run, and the spectra case drives the probe
spectra of include/alis_dev.h.

    dipole     an electric and a magnetic point dipole in a vacuum box with CPML on every face; FP32, and FP64 with eight
               probes read every step: the smallest worlds, where launches and latency count
    scatter    TF/SF scattering by a gold block (Drude pole and two Lorentz pairs) on a dielectric
               half space, with a multi-frequency phaser box around it: the ordinary solve, in FP32
               fields with FP64 DFT sums (the default) and in FP64
    spheres    a lattice of gold spheres in a TF/SF plane wave: many dispersive objects in one world
    array      dielectric pillars on glass, periodic in x and y with CPML in z, plane wave and a
               phaser on the z faces: the largest worlds
    bands      a band sweep: Bloch worlds of a photonic crystal slab at many k points, complex
               fields, all stepped together, eight probes per world read every step
    mix        scattering requests of different sizes stepped together with their phasers, as the
               serving loop does it
    farfield   the (theta, phi) far-field map of an array's phaser, both polarisations
    spectra    the running DFT of many probes, as writeSpectrum keeps one per world

exact() restates the same problems from their definition in double precision: the Yee update with
CPML, trapezoidal ADE currents, Bloch phases, TF/SF strips from an auxiliary world, the surface DFT
and its flux, and the near-to-far projection.
"""
import ctypes
import math
import random
import struct

import numpy as np
import torch

import alis_amd

INF = float(np.finfo(np.float32).max)
PML, PBC, BBC = 3, 4, 6
EV = 1240.0

# ---------------------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------------------


def listed():
    return [
        # the smallest solve: a 40^3 box (10-cell CPML), five launches a step
        {"name": "dipole-40", "kind": "dipole", "cells": 40, "bits": 32, "steps": 400, "probes": 0},
        # the 64^3 FP64 dipole with eight probes (two components each) read every step
        {"name": "dipole-64-fp64-probes", "kind": "dipole", "cells": 64, "bits": 64, "steps": 400, "probes": 8},
        # ordinary scattering solves: a small grid, an odd one in FP64, the 256^3 headline
        {"name": "scatter-128", "kind": "scatter", "cells": 128, "bits": 32, "steps": 600, "dl": 35.0},
        {"name": "scatter-151-fp64", "kind": "scatter", "cells": 151, "bits": 64, "steps": 400, "dl": 35.0},
        {"name": "scatter-256", "kind": "scatter", "cells": 256, "bits": 32, "steps": 700, "dl": 16.5},
        # 64 dispersive objects
        {"name": "spheres-200", "kind": "spheres", "cells": 200, "bits": 32, "steps": 500, "side": 4},
        # the large periodic array: 401 x 401 x 200 nodes
        {"name": "array-400", "kind": "array", "cells": 400, "nz": 200, "bits": 32, "steps": 500},
        # 32 k points of 65 x 65 x 50 nodes, complex fields
        {"name": "bands-32", "kind": "bands", "worlds": 32, "cells": 64, "nz": 50, "bits": 32, "steps": 300},
        # the same in FP64 on an odd, smaller cell
        {"name": "bands-9-fp64", "kind": "bands", "worlds": 9, "cells": 37, "nz": 43, "bits": 64, "steps": 300},
        # requests with grid edges of 64 to 128 stepped together
        {"name": "mix-6", "kind": "mix", "edges": "64,96,64,128,77,96", "bits": 32, "steps": 400},
        # far-field image of 121 x 121 directions from two 321 x 321 faces
        {"name": "farfield-320", "kind": "farfield", "cells": 320, "nz": 72, "bits": 32, "steps": 40, "map": 121},
        # 24 probe spectra (8 probes, 256 bins) over 512 steps
        {"name": "spectra-24", "kind": "spectra", "spectra": 24, "probes": 8, "bins": 256, "steps": 512},
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dipole", "dipole", "scatter", "scatter", "spheres", "array", "bands", "mix", "farfield", "spectra"])
    bits = rng.choice([32, 32, 64])
    if kind == "dipole":
        n = _between(rng, 32, 200)
        return {"kind": kind, "cells": n, "bits": bits, "steps": 400 if n < 128 else 200, "probes": rng.choice([0, 4, 8])}
    if kind == "scatter":
        n = _between(rng, 96, 256 if bits == 32 else 200)
        return {"kind": kind, "cells": n, "bits": bits, "steps": rng.randrange(300, 500), "dl": rng.choice([16.5, 35.0, 60.0])}
    if kind == "spheres":
        return {"kind": kind, "cells": _between(rng, 130, 220), "bits": bits, "steps": rng.randrange(200, 400), "side": rng.choice([2, 3, 4])}
    if kind == "array":
        return {"kind": kind, "cells": 2 * _between(rng, 60, 180), "nz": _between(rng, 72, 180), "bits": 32, "steps": rng.randrange(150, 300)}
    if kind == "bands":
        return {"kind": kind, "worlds": _between(rng, 2, 32 if bits == 32 else 12), "cells": _between(rng, 20, 72), "nz": _between(rng, 36, 72),
                "bits": bits, "steps": rng.randrange(150, 300)}
    if kind == "mix":
        edges = [rng.choice([64, 72, 81, 96, 110, 128]) for _ in range(rng.randrange(2, 8))]
        return {"kind": kind, "edges": ",".join(map(str, edges)), "bits": bits, "steps": rng.randrange(200, 400)}
    if kind == "farfield":
        return {"kind": kind, "cells": 2 * _between(rng, 50, 160), "nz": 72, "bits": 32, "steps": 40, "map": _between(rng, 21, 121)}
    return {"kind": kind, "spectra": _between(rng, 1, 32), "probes": rng.randrange(1, 17), "bins": _between(rng, 40, 600),
            "steps": 256 * rng.randrange(1, 3)}


# ---------------------------------------------------------------------------------------
# The problem of a case: plain numbers that both the API calls and exact() take
# ---------------------------------------------------------------------------------------


def _f32(v):
    return float(np.float32(v))


class _Scene:
    """One world: node extents of the domain and CPML thickness per axis, objects (first ones take
    precedence), sources, TF/SF box and phaser."""
    dt, dx = 1.0, 2.0
    bits = 32
    objects = ()          # (shape, (x0, x1, y0, y1, z0, z1), matter); matter (eps, ((w, r[, f]), ...))
    dipoles = ()          # (component "Ez" or "Hz", (x, y, z), waveform, wavelength, supplement)
    tfsf = None           # (x0, x1, y0, y1, z0, z1) in nm, lit from above by an x-polarised Band wave
    wave = (400.0, 900.0)
    phaser = None         # (LMin, LMax, dL, x0, x1, y0, y1, z0, z1) in nm
    bloch = None          # (fx, fy): phase across the x and y period over 2 pi
    probes = ()

    def __init__(self, lo, hi, pml):
        self.lo, self.hi, self.pml = lo, hi, pml     # pml: CPML cells per axis, 0: periodic

    @property
    def MIN(self):
        return tuple(a - (p + 1 if p else 0) for a, p in zip(self.lo, self.pml))

    @property
    def NUM(self):
        return tuple(b - a + 1 + (2 * (p + 1) if p else 0) for a, b, p in zip(self.lo, self.hi, self.pml))

    @property
    def cells(self):
        return math.prod(self.NUM)


def _cube(cells, pml):
    d = cells - 2 * (pml + 1)
    a = (d - 1) // 2
    return (-a,) * 3, (d - 1 - a,) * 3, (pml,) * 3


def _gold(plasma):
    return (1.5, ((plasma, 0.07, 0.0), (2.6, 0.3, 0.5), (3.5, 0.6, 0.8)))


def _dipole(case, rng):
    s = _Scene(*_cube(case["cells"], 10))
    s.dt, s.dx, s.bits = 5.0, 10.0, case["bits"]
    d = s.hi[0] - s.lo[0]

    def spot(reach):
        return tuple(10.0 * rng.randrange(-int(reach * d), int(reach * d) + 1) for _ in range(3))
    s.dipoles = [(c, spot(0.15), "Pulse", float(rng.randrange(450, 700)), float(rng.randrange(400, 600))) for c in ("Ez", "Hz")]
    s.probes = [spot(0.4) for _ in range(case["probes"])]
    return s


def _scatter(case, rng):
    """Block of half width b cells standing on a half space of index 1.5; TF/SF box 10 cells
    around it, phaser box 10 cells around that (dx = 2 nm)."""
    s = _Scene(*_cube(case["cells"], 16))
    s.bits = case["bits"]
    d = s.hi[0] - s.lo[0] + 1
    b = max(4, d // 8) + rng.randrange(-2, 1)
    w, t, p = 2.0 * b + 0.5, 2.0 * (b + 10), 2.0 * (b + 14)
    s.objects = [("Box", (-w, w, -w, w, 0.5, 2.0 * rng.randrange(b, b + 6) + 0.5), _gold(_f32(rng.uniform(8, 9.5)))),
                 ("Box", (-INF, INF, -INF, INF, -INF, 0.5), (2.25, ()))]
    s.tfsf = (-t, t, -t, t, -t, t)
    s.phaser = (400.0, 900.0, case["dl"], -p, p, -p, p, -p, p)
    return s


def _spheres(case, rng):
    s = _Scene(*_cube(case["cells"], 16))
    s.bits = case["bits"]
    d, side = s.hi[0] - s.lo[0] + 1, case["side"]
    pitch = 2 * ((d - 30) // (2 * side))                                  # cells
    at = [2.0 * pitch * (q - (side - 1) / 2) for q in range(side)]
    s.objects, gold = [], _gold(_f32(rng.uniform(8, 9.5)))
    for x in at:
        for y in at:
            for z in at:
                r = _f32(pitch * rng.uniform(0.5, 0.8))
                s.objects.append(("Ball", (x - r, x + r, y - r, y + r, z - r, z + r), gold))
    t = 2.0 * (pitch * side // 2 + 2)
    s.tfsf = (-t, t, -t, t, -t, t)
    return s


def _array(case, rng):
    """Pillars of eps 6.25 with a pitch near 60 cells on glass, dx = 5 nm."""
    n, nz = case["cells"], case["nz"]
    d = nz - 34
    a = (d - 1) // 2
    s = _Scene((-(n // 2), -(n // 2), -a), (n // 2, n // 2, d - 1 - a), (0, 0, 16))
    s.dt, s.dx, s.bits = 2.5, 5.0, case["bits"]
    side = max(1, n // 60)
    pitch, half, tall = 5.0 * n / side, 2.5 * n, 5.0 * (d // 4) + 1.25
    s.objects = []
    for p in range(side * side):
        x, y = -half + pitch * (p % side + 0.5), -half + pitch * (p // side + 0.5)
        r = pitch * rng.uniform(0.15, 0.3)
        s.objects.append(("RodZ", tuple(map(_f32, (x - r, x + r, y - r, y + r, 1.25, tall))), (6.25, ())))
    s.objects.append(("Box", (-INF, INF, -INF, INF, -INF, 1.25), (2.25, ())))
    zt = 5.0 * (d // 4 + 3)
    s.tfsf = (-half, half, -half, half, -15.0, zt)
    s.phaser = (550.0, 550.0, 550.0, -INF, INF, -INF, INF, -25.0, zt + 15.0)
    return s


def _bands(case, rng):
    """Slab of eps 12 with four air holes, one world per k point along Gamma-X-M; dx = 10 nm."""
    n, nz, nw = case["cells"], case["nz"], case["worlds"]
    d = nz - 18
    a = (d - 1) // 2
    scenes = []
    for q in range(nw):
        t = 2 * (q + rng.uniform(0.2, 0.8)) / nw
        fx, fy = (0.5 * t, 0.0) if t < 1 else (0.5, 0.5 * (t - 1))
        s = _Scene((0, 0, -a), (n, n, d - 1 - a), (0, 0, 8))
        s.dt, s.dx, s.bits, s.bloch = 5.0, 10.0, case["bits"], (_f32(fx), _f32(fy))
        L, r, h = 10.0 * n, _f32(10.0 * n * 0.15 + 0.3), 10.0 * (d // 5) + 2.5
        s.objects = [("RodZ", tuple(map(_f32, (L * u - r, L * u + r, L * v - r, L * v + r, -h, h))), (1.0, ()))
                     for u in (0.25, 0.75) for v in (0.25, 0.75)]
        s.objects.append(("Box", (-INF, INF, -INF, INF, -h, h), (12.0, ())))

        def spot():
            return (10.0 * rng.randrange(2, n - 2), 10.0 * rng.randrange(2, n - 2), 10.0 * rng.randrange(-(d // 4), d // 4 + 1))
        s.dipoles = [("Ez" if p % 2 else "Hz", spot(), "Band", float(rng.randrange(600, 1000)), 2500.0) for p in range(8)]
        s.probes = [spot() for _ in range(8)]
        scenes.append(s)
    return scenes


def _mix(case, rng):
    """Spheres in vacuum as the serving loop's requests: 8-cell CPML, TF/SF box 3 cells and
    phaser box 6 cells around the sphere, 16 wavelengths."""
    scenes = []
    for n in map(int, case["edges"].split(",")):
        s = _Scene(*_cube(n, 8))
        s.bits = case["bits"]
        r = rng.randrange(10, min(40, (n - 20) // 2 - 8) + 1)
        R, t, p = 2.0 * r, 2.0 * (r + 3), 2.0 * (r + 6)
        s.objects = [("Ball", (-R, R) * 3, _gold(_f32(rng.uniform(8, 9.5))))]
        s.tfsf = (-t, t) * 3
        s.phaser = (400.0, 900.0, 35.0) + (-p, p) * 3
        scenes.append(s)
    return scenes


def _scenes(case, seed):
    rng = random.Random("%s %d" % (case["kind"], seed))
    make = {"dipole": _dipole, "scatter": _scatter, "spheres": _spheres, "array": _array, "farfield": _array, "bands": _bands, "mix": _mix}
    s = make[case["kind"]](case, rng)
    return s if isinstance(s, list) else [s]


def _spectra_samples(case, seed):
    """Damped oscillations, as probes record them: values [steps, spectra, probes]."""
    g = np.random.default_rng(seed)
    n, p, m = case["steps"], case["probes"], case["spectra"]
    f, a, ph = g.uniform(0.004, 0.03, (m, p)), g.uniform(0.1, 10, (m, p)), g.uniform(0, 6.28, (m, p))
    t = np.arange(1, n + 1)[:, None, None]
    return np.ascontiguousarray(a * np.exp(-0.002 * t) * np.sin(2 * np.pi * f * t + ph))


# ---------------------------------------------------------------------------------------
# The C API through ctypes (include/alis.h, include/alis_dev.h)
# ---------------------------------------------------------------------------------------

_F, _I, _P, _D, _L = ctypes.c_float, ctypes.c_int, ctypes.c_void_p, ctypes.c_double, ctypes.c_long


def _floats(*names):
    return [(n, _F) for n in names]


class _Dom(ctypes.Structure):
    _fields_ = _floats("x0", "x1", "y0", "y1", "z0", "z1")


class _Sur(ctypes.Structure):
    _fields_ = _floats("x0", "x1", "y0", "y1", "z0", "z1") + [("Num", _I)] + _floats("SigmaMax", "KappaMax", "AlphaMax", "SigmaPower", "AlphaPower")


class _Nug(ctypes.Structure):
    _fields_ = [("m", _I), ("Min", _F), ("Max", _F)]


class _Res(ctypes.Structure):
    _fields_ = _floats("dt", "dx", "dy", "dz", "eV") + [("subN", _I), ("nug", _Nug * 3), ("gridFunction", _P * 3)]


class _Matter(ctypes.Structure):
    _fields_ = [("e", _F * 3), ("P", _F * 4 * 6), ("d", _F * 6 * 3)]


class _Object(ctypes.Structure):
    _fields_ = [("S", _P), ("f", _F * 3 * 3), ("p", _P)]


class _VField(ctypes.Structure):
    _fields_ = [("f", _P * 3), ("psi", _P * 12), ("J", _P * 6), ("t", _F)]


class _World(ctypes.Structure):
    _fields_ = ([("Dom", _Dom), ("Res", _Res), ("Sur", _Sur)] + [("scale", _F * 7), ("bounds", _F * 12), ("phases", _F * 10), ("sizes", _F * 6)]
                + [("node", _I * 9), ("NODE", _I * 9), ("surfaces", _I * 6), ("subN", _I), ("complexField", _I), ("sourceType", _I)]
                + [("n", ctypes.c_ulong), ("N", ctypes.c_ulong), ("T", ctypes.c_ulong), ("maps", _P * 6), ("ID", ctypes.c_char * 128)]
                + [("E", ctypes.POINTER(_VField)), ("H", ctypes.POINTER(_VField))])


class _Phaser(ctypes.Structure):
    _fields_ = [("W", _P), ("box", _I * 6), ("kMIN", _I), ("xNUM", _I), ("yNUM", _I), ("N", ctypes.c_ulong), ("f", _F), ("A", _F),
                ("dE", _P), ("dH", _P), ("expik", _F * 4), ("ex", _P), ("ez", _P), ("faces", _P * 36), ("count", _I), ("devId", _I),
                ("hostStale", _I), ("view", _P), ("viewValid", _I), ("faceFlux", _P), ("faceFluxValid", _I)]


class _Slice(ctypes.Structure):
    _fields_ = [("range", _I * 6), ("RANGE", _I * 9), ("C", _P), ("F", _P), ("interpolate", _P)]


_METHOD = ctypes.CFUNCTYPE(None, _P, ctypes.POINTER(_Slice), _F, ctypes.c_char_p, ctypes.c_char_p, _P)
_bound = None


def _lib():
    global _bound
    if _bound is None:
        lib = alis_amd.library()
        for name, res, args in (
                ("createWorld", _P, [_Dom, _Res, _Sur, ctypes.c_char_p]), ("deleteWorld", None, [_P]),
                ("putObjectArray", None, [_P, _P, _P]), ("worldPrecision", None, [_P, _I, _I]),
                ("pointDipole", None, [_P, _P, _F, _F, _F, _P, _F, _F, _F, _F]),
                ("planewave", None, [_P, _Dom, _P, _F, _F, _P, _F, _F, _F, _F]),
                ("createPhasers", _P, [_P] + [_F] * 9), ("deletePhaser", None, [_P]),
                ("updateE", None, [_P]), ("updateH", None, [_P]), ("updatePhaser", None, [_P, _P]),
                ("updateWorldsE", None, [_P, _I]), ("updateWorldsH", None, [_P, _I]), ("updatePhaserArrays", None, [_P, _P, _I]),
                ("syncWorld", None, [_P]), ("get", _F, [_P, _P, _F, _F, _F]), ("phaserPoyntingOut", _F, [_P]),
                ("farFieldProfile", None, [_P, _P, _P, _I, _I, _METHOD, ctypes.c_char_p]),
                ("alis_dev_spectrum_create", _I, [_I, _I, _I, ctypes.POINTER(_P)]), ("alis_dev_spectrum_add", _I, [_P, _D, _P]),
                ("alis_dev_spectrum_read", _I, [_P, _P]), ("alis_dev_spectrum_release", None, [_P])):
            f = getattr(lib, name)
            f.restype, f.argtypes = res, args
        _bound = lib
    return _bound


def _entry(name):
    return ctypes.cast(getattr(_lib(), name), _P)


def _host_array(f, MIN, NUM, owner):
    """The cells MIN .. MIN+NUM-1 of a float*** over the grid and its ghost layer; the array
    keeps the world that holds the memory."""
    base = f
    for m in MIN[:2]:
        base = _P.from_address(base + 8 * (m - 1)).value
    base += 4 * (MIN[2] - 1)
    shape = tuple(n + 2 for n in NUM)
    memory = (ctypes.c_float * math.prod(shape)).from_address(base)
    memory.owner = owner
    return np.ctypeslib.as_array(memory).reshape(shape)[1:-1, 1:-1, 1:-1]


class _Solve:
    """A world built through the API and its phaser."""

    def __init__(self, s):
        lib, self.scene = _lib(), s
        self.W = self.P = None
        dx = s.dx
        z = [c for ax in range(3) for c in (s.lo[ax] * dx, s.hi[ax] * dx)]
        r = _Res(dt=s.dt, dx=dx, eV=EV, subN=1)
        u = _Sur(Num=max(s.pml))
        for a, n in enumerate("xyz"):
            setattr(u, n + "0", PML if s.pml[a] else BBC if s.bloch else PBC)
            if s.bloch and a < 2:
                setattr(u, n + "1", (s.hi[a] - s.lo[a]) * dx / s.bloch[a] if s.bloch[a] else INF)
        self.W = lib.createWorld(_Dom(*z), r, u, b"")
        if s.objects:
            m, o = (_Matter * (len(s.objects) + 1))(), (_Object * (len(s.objects) + 1))()
            for q, (shape, box, (eps, poles)) in enumerate(s.objects):
                m[q].e[0], o[q].S = eps, _entry(shape)
                for a in range(6):
                    o[q].f[a // 2][a % 2] = box[a]
                for p, pole in enumerate(poles):
                    for v, x in enumerate(pole):
                        m[q].P[p][v] = x
            m[len(s.objects)].e[0] = 1.0
            lib.putObjectArray(self.W, m, o)
            self.keep = m, o
        for comp, (x, y, zz), wave, length, sup in s.dipoles:
            lib.pointDipole(self.W, _entry(comp), x, y, zz, _entry(wave), length, sup, 0.0, 0.0)
        if s.tfsf:
            lib.planewave(self.W, _Dom(*s.tfsf), _entry("Ppol"), 0.0, 0.0, _entry("Band"), s.wave[0], s.wave[1], 0.0, 0.0)
        if s.phaser:
            self.P = lib.createPhasers(self.W, *s.phaser)
        lib.worldPrecision(self.W, s.bits, 64)
        self.freqs = _Phaser.from_address(self.P).count if self.P else 0

    def fields(self):
        """The host fields (E x y z, H x y z; the imaginary parts of a Bloch world after them)."""
        _lib().syncWorld(self.W)
        w, s = _World.from_address(self.W), self.scene
        return [_host_array(V[m].f[a], s.MIN, s.NUM, self) for m in range(1 + w.complexField) for V in (w.E, w.H) for a in range(3)]

    def flux(self):
        out, size = _lib().phaserPoyntingOut, ctypes.sizeof(_Phaser)
        return np.array([out(self.P + size * q) for q in range(self.freqs)], dtype=np.float32)

    def __del__(self):
        if _bound and self.P:
            _bound.deletePhaser(self.P)
        if _bound and self.W:
            _bound.deleteWorld(self.W)


class _Spectra:
    def __init__(self, case, seed):
        self.v = _spectra_samples(case, seed)
        self.case, self.n, self.h = case, 0, []
        for _ in range(case["spectra"]):
            h = _P()
            if _lib().alis_dev_spectrum_create(case["probes"], case["bins"], _top(case), ctypes.byref(h)):
                raise RuntimeError(_lib().alis_dev_error().decode())
            self.h.append(h)

    def __del__(self):
        for h in self.h if _bound else ():
            _bound.alis_dev_spectrum_release(h)


def _top(case):
    return case["bins"] + 40


def _tau(case, n):
    return n / (4.0 * case["bins"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "spectra":
        return _Spectra(case, seed)
    solves = [_Solve(s) for s in _scenes(case, seed)]
    state = {"case": case, "solves": solves}
    if kind in ("bands", "mix"):
        state["W"] = (_P * len(solves))(*[q.W for q in solves])
        state["P"] = (_P * len(solves))(*[q.P for q in solves])
    if kind == "farfield":
        _march(state)                     # the run whose far field is wanted
    return state


def _march(state):
    """The steps of a pass; the probe values read on the way, in order."""
    lib, case, solves = _lib(), state["case"], state["solves"]
    read = []
    if "W" in state:
        n, W, P = len(solves), state["W"], state["P"]
        E, H, many, get = lib.updateWorldsE, lib.updateWorldsH, lib.updatePhaserArrays, lib.get
        at = [(q.W, _entry("Ez" if p % 2 else "Hz"), *x) for q in solves for p, x in enumerate(q.scene.probes)]
        phasers = case["kind"] == "mix"
        for _ in range(case["steps"]):
            E(W, n)
            H(W, n)
            if phasers:
                many(W, P, n)
            for a in at:
                read.append(get(*a))
        return read
    W, P, E, H, update, get = solves[0].W, solves[0].P, lib.updateE, lib.updateH, lib.updatePhaser, lib.get
    at = [(W, _entry(c), *x) for x in solves[0].scene.probes for c in ("Ez", "Hy")]
    for _ in range(case["steps"]):
        E(W)
        H(W)
        if P:
            update(W, P)
        for a in at:
            read.append(get(*a))
    return read


def run(state):
    lib = _lib()
    if isinstance(state, _Spectra):
        add, base, stride = lib.alis_dev_spectrum_add, state.v.ctypes.data, 8 * state.case["probes"]
        for n in range(state.case["steps"]):
            state.n += 1
            tau = _tau(state.case, state.n)
            for h in state.h:
                add(h, tau, base)
                base += stride
        out = np.empty((len(state.h), state.case["probes"], state.case["bins"], 2))
        for q, h in enumerate(state.h):
            lib.alis_dev_spectrum_read(h, out[q].ctypes.data)
        return out
    case, solves = state["case"], state["solves"]
    if case["kind"] == "farfield":
        maps, n = {}, case["map"]

        def keep(W, S, most, field, name, cmap):
            f = S.contents.F
            data = _P.from_address(_P.from_address(f).value).value
            maps[name.decode().rsplit("ff-", 1)[-1]] = np.ctypeslib.as_array((ctypes.c_float * (n * n)).from_address(data)).reshape(n, n).copy()
        lib.farFieldProfile(solves[0].W, solves[0].P, _entry("CylindericalMap"), n, n, _METHOD(keep), b"ff-")
        return maps
    read = _march(state)
    out = {}
    if read:
        out["probes"] = np.array(read, dtype=np.float32)
    # a band sweep looks at the fields of a few of its k points, the other programs at all
    for q in solves if case["kind"] != "bands" else solves[::max(1, -(-len(solves) // 4))]:
        out.setdefault("fields", []).append(q.fields())
    if solves[0].P:
        out["flux"] = [q.flux() for q in solves]
    return out


def work(case):
    """Per step and cell the six field values read and written once, 1/eps read once where there
    are objects, each CPML slab value read and written once; per phaser update four values a face
    cell; the fields taken home at the end.  Spectra and far field: samples, faces and results."""
    kind = case["kind"]
    if kind == "spectra":
        n = case["spectra"] * case["probes"] * case["bins"]
        return {"bytes": 8.0 * case["steps"] * case["spectra"] * (case["probes"] + 1) + 32.0 * n, "flops": 4.0 * n * case["steps"]}
    if kind == "farfield":
        n, d = (case["cells"] + 1) ** 2, case["map"] ** 2
        return {"bytes": 2.0 * 4 * n * 16 + 7 * 4 * d, "flops": 8.0 * 8 * n * d}
    total = flops = 0.0
    for s in _scenes(case, 0):
        size, parts = s.bits // 8, 2 if s.bloch else 1
        slab = sum(2 * s.pml[a] * s.cells / s.NUM[a] for a in range(3))
        total += case["steps"] * size * (parts * (12 * s.cells + 2 * 4 * slab) + (3 * s.cells if s.objects else 0))
        flops += case["steps"] * parts * s.cells * 36.0
        if s.phaser:
            total += case["steps"] * size * 4.0 * sum(len(f) for f in _face_cells(s))
        total += 6 * parts * 4.0 * s.cells                      # the fields taken home
    return {"bytes": total, "flops": flops}


def _face_cells(s):
    b = _phaser_box(s)
    n = [hi - lo + 1 for lo, hi in b]
    return [range(n[(a + 1) % 3] * n[(a + 2) % 3]) for a in range(3) if s.pml[a] for _ in range(2)]


# ---------------------------------------------------------------------------------------
# The same problems in double precision
# ---------------------------------------------------------------------------------------


def _band(length, sup, dt):
    res = math.ceil(1.25 * sup / length + 0.5) if sup > length else 2
    dev = 2 * math.pi / length / (res - 0.5)
    peak = math.floor(length * (res - 0.5) / dt) * dt

    def f(t):
        x = (t - peak) * dev
        return 0.0 if t == peak else 2 * (math.cos(x * res) - math.cos(x)) / x
    return f, int(2 * length * (res - 0.5) / dt)


def _pulse(length, sup, dt):
    dev = 2 * length * length / (math.pi * sup)
    half = math.floor(math.pi * dev / dt)

    def f(t):
        return math.sin(2 * math.pi / length * (t - half * dt)) * math.exp(-((t - half * dt) / dev) ** 2)
    return f, 2 * half


def _inside(shape, box, x, y, z):
    """The shape's points among float32 coordinates (its inequality is evaluated in float32)."""
    b = [np.float32(v) for v in box]

    def unit(v, lo, hi):
        u = (np.float32(2) * v - lo - hi) / (hi - lo)
        return u * u
    if shape == "Ball":
        return unit(x, b[0], b[1]) + unit(y, b[2], b[3]) + unit(z, b[4], b[5]) < 1
    zin = (b[4] <= z) & (z <= b[5])
    if shape == "RodZ":
        return zin & (unit(x, b[0], b[1]) + unit(y, b[2], b[3]) < 1)
    return (b[0] <= x) & (x <= b[1]) & (b[2] <= y) & (y <= b[3]) & zin


def _owner(s, objects, axis):
    """Index of the object that holds each E position of a component, len(objects) for none."""
    x, y, z = (np.float32(s.dx) * (np.arange(s.NUM[a], dtype=np.float32) + np.float32(s.MIN[a] - (0.5 if a == axis else 0))) for a in range(3))
    own = np.full(s.NUM, len(objects), dtype=np.int16)
    for q in range(len(objects) - 1, -1, -1):
        shape, box, _ = objects[q]
        at = []
        for a, c in enumerate((x, y, z)):
            hit = np.nonzero((c >= box[2 * a]) & (c <= box[2 * a + 1]))[0]
            at.append(slice(hit[0], hit[-1] + 1) if len(hit) else slice(0, 0))
        part = own[at[0], at[1], at[2]]
        if part.size:
            part[np.broadcast_to(_inside(shape, box, x[at[0], None, None], y[None, at[1], None], z[None, None, at[2]]), part.shape)] = q
    return own


class _Yee:
    """One Yee grid (or a batch of Bloch ones on one geometry) in float64 / complex128.  Arrays
    carry a ghost layer; index 1 of an axis is node MIN."""

    def __init__(self, scenes, device, objects=None):
        s = self.s = scenes[0]
        self.dev, self.r, self.dt, self.n, self.t = device, s.dt / s.dx, s.dt, 0, [0.0, 0.0]
        kind = torch.complex128 if s.bloch else torch.float64
        shape = (len(scenes),) + tuple(n + 2 for n in s.NUM)
        self.F = [[torch.zeros(shape, dtype=kind, device=device) for _ in range(3)] for _ in range(2)]
        self.phase = [None, None, None]
        if s.bloch:
            for a in range(2):
                k = torch.tensor([2 * math.pi * q.bloch[a] for q in scenes], dtype=torch.float64, device=device)
                self.phase[a] = torch.polar(torch.ones_like(k), k).reshape(-1, 1, 1, 1)
        self.c, self.ade = None, []
        objects = s.objects if objects is None else objects
        if objects:
            own = [_owner(s, objects, a) for a in range(3)]
            eps = np.array([m[0] for _, _, m in objects] + [1.0])
            self.c = [torch.from_numpy(1 / eps[o]).to(device) for o in own]
            self._currents(objects, own, shape[0], kind)
        self.slabs = [[self._slab(h, f, kind, shape[0]) for f in range(6) if s.pml[f % 3]] for h in range(2)]
        self.sources = [[], []]
        self.aux = None

    def _currents(self, objects, own, nb, kind):
        for matter in sorted({m for _, _, m in objects if m[1]}):
            which = [q for q, o in enumerate(objects) if o[2] == matter]
            hit = np.stack([np.isin(o, which) for o in own])
            at = np.nonzero(hit.any(0))
            box = tuple(slice(int(v.min()), int(v.max()) + 1) for v in at)
            fill = [torch.from_numpy(hit[a][box].astype(np.float64)).to(self.dev) for a in range(3)]
            zero = torch.zeros((nb,) + tuple(fill[0].shape), dtype=kind, device=self.dev)
            u = math.pi * self.dt / EV
            poles = []
            for w, r, f in matter[1]:
                if not f:
                    poles.append(((1 - u * r) / (1 + u * r), 0.0, (2 * u * w) ** 2 / (1 + u * r) / matter[0], None))
                    continue
                g = complex(r, w)
                a, b = (1 - u * g) / (1 + u * g), -g * (1j * f * w) * (2 * u) ** 2 / (1 + u * g) / matter[0]
                poles.append((a.real, -a.imag, b.real, (a.imag / a.real, a.imag ** 2 / a.real + a.real, -b.real * a.imag / a.real + b.imag)))
            # J' = JJ J + JK K + JE E (K' of the pair: KJ J' + KK K + KE E)
            state = [[[zero.clone(), None if p[3] is None else zero.clone()] for p in poles] for _ in range(3)]
            self.ade.append((tuple(slice(b.start + 1, b.stop + 1) for b in box), fill, poles, state))

    def _slab(self, h, face, kind, nb):
        ax, N, n = face % 3, self.s.pml[face % 3], self.s.NUM[face % 3]
        q = np.arange(1, N + 1)
        idx = (N - q + h if face < 3 else n - 1 - N + q)            # cell of depth q
        x = (q - 0.5 * h) / N
        sig = 0.8 * 4.5 * x ** 3.5 * self.r
        order = np.argsort(idx)
        lo = int(idx[order][0])
        view = [1, 1, 1, 1]
        view[1 + ax] = N
        b, d = (torch.from_numpy(np.ascontiguousarray(v[order])).to(self.dev).reshape(view) for v in ((1 - sig / 2) / (1 + sig / 2), self.r * sig / (1 + sig / 2)))
        shape = [nb] + list(self.s.NUM)
        shape[1 + ax] = N
        return ax, slice(lo, lo + N), b, d, torch.zeros(shape, dtype=kind, device=self.dev), torch.zeros(shape, dtype=kind, device=self.dev)

    @staticmethod
    def _at(F, axis=None, d=0):
        i = [slice(None)] + [slice(1, -1)] * 3
        if axis is not None:
            i[1 + axis] = slice(1 + d, F.shape[1 + axis] - 1 + d)
        return F[tuple(i)]

    def curl(self, h):
        G, F, d = self.F[1 - h], self.F[h], 1 if h == 0 else -1
        c = self.c if h == 0 and self.c is not None else (1.0, 1.0, 1.0)
        if h == 0:
            for box, _, _, state in self.ade:
                for a in range(3):
                    for J, _ in state[a]:
                        F[a][(slice(None),) + box] -= J
        for a in range(3):
            b, e = (a + 1) % 3, (a + 2) % 3
            # F_a += c_a dt/d (G_b - G_b(+e) + G_e(+b) - G_e)
            u = self._at(G[b]) - self._at(G[b], e, d)
            u += self._at(G[e], b, d)
            u -= self._at(G[e])
            self._at(F[a]).add_(u * (c[a] * self.r))
        for ax, at, b, k, pa, pb in self.slabs[h]:
            i = [slice(None)] * 4
            i[1 + ax] = at
            i, u, v = tuple(i), (ax + 1) % 3, (ax + 2) % 3
            pa.mul_(b).sub_(k * (self._at(G[v]) - self._at(G[v], ax, d))[i])
            pb.mul_(b).add_(k * (self._at(G[u]) - self._at(G[u], ax, d))[i])
            self._at(F[u])[i] += pa * (c[u][i[1:]] if self.c is not None and h == 0 else 1.0)
            self._at(F[v])[i] += pb * (c[v][i[1:]] if self.c is not None and h == 0 else 1.0)
        if h == 1:
            for box, fill, poles, state in self.ade:
                for a in range(3):
                    e = self.F[0][a][(slice(None),) + box] * fill[a]
                    for (JJ, JK, JE, pair), JKs in zip(poles, state[a]):
                        J, K = JKs
                        J.mul_(JJ).add_(e, alpha=JE)
                        if pair:
                            J.add_(K, alpha=JK)
                            K.mul_(pair[1]).add_(J, alpha=pair[0]).add_(e, alpha=pair[2])

    def ghosts(self, h):
        F, n = self.F[h], self.s.NUM

        def put(comp, ax, to, frm, up, wide):
            dst, src = [slice(None)] * 4, [slice(None)] * 4
            for a in range(3):
                dst[1 + a] = src[1 + a] = slice(1, 2 + n[a] if a in wide else 1 + n[a])
            dst[1 + ax], src[1 + ax] = slice(to, to + 1), slice(frm, frm + 1)
            v = F[comp][tuple(src)]
            if self.phase[ax] is not None:
                v = v * (self.phase[ax] if up else self.phase[ax].conj())
            F[comp][tuple(dst)] = v
        alt = [1 if p else m - 1 for p, m in zip(self.s.pml, n)]
        up = [(m + 1, m + 1 - q) for m, q in zip(n, alt)]           # ghost beyond the last node
        if h == 0:
            for comp, ax in ((0, 0), (2, 2), (1, 1)):
                put(comp, ax, *up[ax], True, ())
            return
        for ax, comps, wide in ((0, (1, 2), (1, 2)), (2, (0, 1), (0, 1))):
            for comp in comps:
                put(comp, ax, *up[ax], True, wide)
        for ax, comps, wide in ((0, (1, 2), (1, 2)), (2, (0, 1), (0, 1))):
            for comp in comps:
                put(comp, ax, 1, 1 + alt[ax], False, wide)
        for comp in (2, 0):
            put(comp, 1, *up[1], True, (0, 2))
        for comp in (2, 0):
            put(comp, 1, 1, 1 + alt[1], False, (0, 2))

    def strips(self, h):
        """Total-field corrections on the box faces (nodes lo..hi of the box) from the auxiliary
        world, whose x and y rows repeat beyond its own two."""
        A, s, (lo, hi) = self.aux, self.s, self.box
        MIN, MAX = s.MIN, tuple(m + n - 1 for m, n in zip(s.MIN, s.NUM))
        inner = [(a if a == m else a + 1, b + 1 if b == M else b) for a, b, m, M in zip(lo, hi, MIN, MAX)]
        alt = ((1, 0, 0, 0, 1, 1), (0, 1, 0, 1, 0, 1))
        for ax in range(3):
            u, v = (ax + 1) % 3, (ax + 2) % 3
            for side in (0, 1):
                if lo[ax] <= MIN[ax] if side == 0 else hi[ax] >= MAX[ax]:
                    continue
                at = lo[ax] if side == 0 else hi[ax] + h
                sign = (1 if side else -1) * (-1 if h else 1)
                # F_v from G_u with one sign, F_u from G_v with the other
                for fa, ga, sg in ((v, u, sign), (u, v, -sign)):
                    rng, src = [None] * 3, [None] * 3
                    for a in range(3):
                        if a == ax:
                            rng[a] = (at, at)
                        elif (a == fa) == (h == 0):
                            rng[a] = inner[a]
                        else:
                            rng[a] = (lo[a], hi[a])
                        i = np.arange(rng[a][0], rng[a][1] + 1) + ((1 if h == 0 else -1) if a == ax and side else 0)
                        if a < 2:
                            last = A.s.MIN[a] + 1
                            i = np.where(i > last, last + alt[a][(1 - h) * 3 + ga], i)
                        src[a] = torch.from_numpy(i - A.s.MIN[a] + 1).to(self.dev)
                    g = A.F[1 - h][ga][0][src[0][:, None, None], src[1][None, :, None], src[2][None, None, :]]
                    cut = tuple(slice(a - m, b - m + 1) for (a, b), m in zip(rng, MIN))
                    if h == 0 and self.c is not None:
                        # 1/eps; a strip may reach the ghost plane, where the medium continues
                        cc = self.c[fa][tuple(slice(c.start, min(c.stop, n)) for c, n in zip(cut, s.NUM))]
                        for a in range(3):
                            if cc.shape[a] < g.shape[a]:
                                cc = torch.cat([cc, cc.narrow(a, cc.shape[a] - 1, 1)], a)
                        g = g * cc
                    self.F[h][fa][(slice(None),) + tuple(slice(c.start + 1, c.stop + 1) for c in cut)] += sg * self.r * g

    def half(self, h):
        self.curl(h)
        if self.aux:
            self.aux.half(h)
            self.strips(h)
        t = self.t[1 - h]
        n = self.n
        for index, amp, wave, last in self.sources[h]:
            if n < last:
                self.F[h][index[0]][index[1]] += amp * wave(t)
        self.ghosts(h)
        if h == 0:
            self.n += 1
            self.t[0] = self.n * self.dt
        else:
            self.t[1] = self.t[0] + 0.5 * self.dt


def _node(s, x):
    return int(round(x / s.dx))


def _phaser_box(s):
    return [(max(s.lo[a], _node(s, max(s.phaser[3 + 2 * a], -1e6))), min(s.hi[a], _node(s, min(s.phaser[4 + 2 * a], 1e6)))) for a in range(3)]


def _grid(scenes, device):
    """The grid of a case with its sources and auxiliary world."""
    g, s = _Yee(scenes, device), scenes[0]
    for q, w in enumerate(scenes):
        for comp, at, wave, length, sup in w.dipoles:
            f, last = (_band if wave == "Band" else _pulse)(length, sup, s.dt)
            h, axis = (0 if comp[0] == "E" else 1), "xyz".index(comp[1])
            amp = math.sqrt(1.5 / math.pi) * length / s.dt ** 2 * g.r ** 3 * (0.5 if h == 0 else 0.25)
            i = [_node(s, v) - m + 1 for v, m in zip(at, s.MIN)]
            wide = [a == axis if h == 0 else a != axis for a in range(3)]
            box = tuple(slice(c, c + 1 + k) for c, k in zip(i, wide))
            if h == 0 and g.c is not None:
                amp = amp * g.c[axis][tuple(slice(b.start - 1, b.stop - 1) for b in box)]
            g.sources[h].append(((axis, (q,) + box), amp, f, last))
    if s.tfsf:
        lo, hi = [], []
        for a in range(3):
            x0, x1 = _node(s, s.tfsf[2 * a]), _node(s, s.tfsf[2 * a + 1])
            lo.append(x0 if x0 >= s.lo[a] else s.MIN[a])
            hi.append(x1 if x1 <= s.hi[a] else s.MIN[a] + s.NUM[a] - 1)
        g.box = (lo, hi)
        x = _Scene((s.MIN[0], s.MIN[1], s.lo[2] - 1), (s.MIN[0] + 1, s.MIN[1] + 1, s.hi[2] + 1), (0, 0, 12))
        x.dt, x.dx = s.dt, s.dx
        g.aux = _Yee([x], device, [o for o in s.objects if o[1][0] == -INF])
        f, last = _band(*s.wave, s.dt)
        top = s.hi[2] + 1 - x.MIN[2] + 1
        every = (0, slice(1, -1), slice(1, -1))
        g.aux.sources[0].append(((0, every + (top,)), g.r, f, last))
        g.aux.sources[1].append(((1, every + (top + 1,)), -g.r, f, last))
    return g


class _Surface:
    """The phaser's running DFT on the faces with CPML beyond them."""

    def __init__(self, g):
        s = self.s = g.s
        lmin, lmax, dl = s.phaser[:3]
        nmin, nmax = math.floor(lmin / dl), math.ceil(lmax / dl)
        self.f = torch.tensor([(nmax - n) / (dl * nmin * nmax) for n in range(nmax - nmin + 1)], dtype=torch.float64, device=g.dev)
        wave, last = _band(*s.wave, s.dt)
        t = torch.arange(1, last, dtype=torch.float64, device=g.dev) * s.dt
        w = torch.tensor([wave(v) for v in t.tolist()], dtype=torch.float64, device=g.dev)
        self.A = 1 / (w * torch.exp(2j * math.pi * self.f[:, None] * t)).sum(1).abs()
        self.box = _phaser_box(s)
        self.faces = {}
        for ax in range(3):
            if s.pml[ax]:
                for side in (0, 1):
                    self.faces[ax, side] = [0.0] * 4

    def cells(self, ax, side, up=0):
        i = [slice(a - m + 1, b - m + 2) for (a, b), m in zip(self.box, self.s.MIN)]
        i[ax] = self.box[ax][side] - self.s.MIN[ax] + 1 + up
        return (0,) + tuple(i)

    def add(self, g):
        e, h = (torch.exp(2j * math.pi * self.f * t).reshape(-1, 1, 1) for t in g.t)
        for (ax, side), acc in self.faces.items():
            i, up = self.cells(ax, side), self.cells(ax, side, 1)
            for q, c in enumerate(((ax + 1) % 3, (ax + 2) % 3)):
                acc[q] = acc[q] + e * g.F[0][c][i]
                acc[2 + q] = acc[2 + q] + h * (0.5 * (g.F[1][c][i] + g.F[1][c][up]))

    def flux(self):
        total = 0.0
        for (ax, side), acc in self.faces.items():
            # face arrays run over the two other axes in x, y, z order
            rest = [a for a in range(3) if a != ax]
            u, v = (ax + 1) % 3, (ax + 2) % 3
            for e, h, along, sg in ((acc[0], acc[3], v, 1), (acc[1], acc[2], u, -1)):
                p = (e * h.conj()).real
                d = 1 + rest.index(along)                     # trapezoid axis; the other drops its first cell
                w = torch.full((p.shape[d],), self.s.dx, dtype=torch.float64, device=p.device)
                w[0] *= 0.5
                w[-1] *= 0.5
                o = 3 - d
                p = p.narrow(o, 1, p.shape[o] - 1) * (w.reshape(1, -1, 1) if d == 1 else w.reshape(1, 1, -1))
                total = total + (1 if side else -1) * sg * self.s.dx * p.sum((1, 2))
        return total * self.A ** 2


def _far(surface, n):
    """The n x n cylindrical map of a z-face phaser over an x-y periodic array in layers."""
    s, dev = surface.s, surface.f.device
    f = float(surface.f[0])
    (i0, i1), (j0, j1), (k0, k1) = surface.box
    x, y = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    th, ph = np.float32(180.0 - 180.0 * y / n).astype(np.float64).ravel(), np.float32(360.0 * x / n).astype(np.float64).ravel()
    graze = (89 < th) & (th < 91)
    cols = np.concatenate([np.nonzero(~graze)[0], np.nonzero(graze)[0], np.nonzero(graze)[0]])
    ng = int(graze.sum())
    m = len(th) - ng
    theta = th[cols].copy()
    theta[m:m + ng], theta[m + ng:] = 89.0, 91.0
    weight = np.where(graze[cols], 0.5, 1.0)
    # the medium along z at the corner of the phaser box, one node past it
    k = np.arange(k0, k1 + 2)
    layer = [o for o in s.objects if o[0] == "Box"][0]
    ex = np.where(np.float32(s.dx) * k.astype(np.float32) <= np.float32(layer[1][5]), layer[2][0], 1.0)
    ez = np.where(np.float32(s.dx) * (k - 0.5).astype(np.float32) <= np.float32(layer[1][5]), layer[2][0], 1.0)
    sn, dz = np.sin(np.pi * f * s.dt), s.dx / s.dt        # cell width over dt
    K = len(k)
    up = theta < 90
    edge = np.where(up, ex[K - 2], ex[0])
    sth = np.sin(theta * np.pi / 180) * np.sqrt(edge)
    s2 = sth ** 2
    E, H = {}, {}
    for pol in "PS":
        e, h = np.zeros((K, len(theta)), complex), np.zeros((K, len(theta)), complex)
        for sel, ks in ((up, range(K - 1)), (~up, range(K - 2, -1, -1))):
            q, b = s2[sel], (0 if ks.start == 0 else K - 1)
            root = np.sqrt(ex[b] - q + 0j)
            turn = np.arcsin(sn * root * dz)
            if pol == "P":
                sg = 1 if b else -1
                hh, ee = np.full(q.shape, sg, complex), np.sqrt((1 - q / ez[b] + 0j) / ex[b]) * np.exp(1j * sg * turn)
            else:
                sg = 1 if b else -1
                hh, ee = -sg * root, np.exp(1j * sg * turn)
            te, tn = np.zeros((K, sel.sum()), complex), np.zeros((K, sel.sum()), complex)
            te[b], tn[b] = ee, hh
            for p in ks:
                if pol == "P" and not b:
                    tn[p + 1] = tn[p] + 2j * sn * dz * te[p] * ex[p]
                    te[p + 1] = te[p] + 2j * sn * dz * tn[p + 1] * (1 - q / ez[p + 1])
                elif pol == "P":
                    te[p] = te[p + 1] - 2j * sn * dz * tn[p + 1] * (1 - q / ez[p + 1])
                    tn[p] = tn[p + 1] - 2j * sn * dz * te[p] * ex[p]
                elif not b:
                    tn[p + 1] = tn[p] - 2j * sn * dz * te[p] * (ex[p] - q)
                    te[p + 1] = te[p] - 2j * sn * dz * tn[p + 1]
                else:
                    te[p] = te[p + 1] + 2j * sn * dz * tn[p + 1]
                    tn[p] = tn[p + 1] + 2j * sn * dz * te[p] * (ex[p] - q)
                big = np.abs(tn).max(0) > 1e10
                te[:, big] /= 1e10
                tn[:, big] /= 1e10
            e[:, sel], h[:, sel] = te, tn
        a = np.where(up, K - 2, 0)
        c = np.arange(len(theta))
        mean, root, cth = 0.5 * (h[a, c] + h[a + 1, c]), np.sqrt(edge), np.cos(theta * np.pi / 180)
        out = mean / root - e[a, c] / cth if pol == "P" else e[a, c] + mean / (root * cth)
        norm = np.sqrt(np.sqrt(edge)) / np.abs(out)
        E[pol], H[pol] = e * norm, h * norm
    # in-plane phases and the four sums of each face
    phi = ph[cols]
    kx, ky = (torch.from_numpy(-2 * np.pi * f * sth * t).to(dev) for t in (np.cos(phi * np.pi / 180), np.sin(phi * np.pi / 180)))

    def phases(lo, hi, wave, half):
        pos = (torch.arange(lo, hi + 1, dtype=torch.float64, device=dev) - (0.5 if half else 0)) * s.dx
        w = torch.full_like(pos, s.dx)
        if half:
            w[0] = 0
        else:
            w[0] *= 0.5
            w[-1] *= 0.5
        return w[:, None] * torch.exp(1j * pos[:, None] * wave)
    XN, XH, YN, YH = phases(i0, i1, kx, 0), phases(i0, i1, kx, 1), phases(j0, j1, ky, 0), phases(j0, j1, ky, 1)
    cp, sp = np.cos(phi * np.pi / 180), np.sin(phi * np.pi / 180)
    amp = {}
    for pol in "PS":
        total = 0
        for side in (0, 1):
            F = [v[0] for v in surface.faces[2, side]]
            S = [((F[q] @ (YN if q in (0, 3) else YH)) * (XH if q in (0, 3) else XN)).sum(0).cpu().numpy() for q in range(4)]
            at = K - 2 if side else 0
            e, hm = E[pol][at], 0.5 * (H[pol][at] + H[pol][at + 1])
            tex, tey, thx, thy = (e * cp, e * sp, -hm * sp, hm * cp) if pol == "P" else (-e * sp, e * cp, hm * cp, hm * sp)
            v = S[0] * thy - S[3] * tex - S[1] * thx + S[2] * tey
            total = total + (v if side else -v)
        a = np.zeros(len(th), complex)
        np.add.at(a, cols, weight * total * float(surface.A[0]) * f)
        amp[pol] = a
    p, q = amp["P"], amp["S"]
    c, d = np.cos(ph * np.pi / 180), np.sin(ph * np.pi / 180)
    maps = {"X-pol": abs(p * c - q * d) ** 2, "Y-pol": abs(q * c + p * d) ** 2, "P-pol": abs(p) ** 2, "S-pol": abs(q) ** 2,
            "CL-pol": (p.real + q.imag) ** 2 + (p.imag - q.real) ** 2, "CR-pol": (p.real - q.imag) ** 2 + (p.imag + q.real) ** 2}
    maps["Unpol"] = maps["P-pol"] + maps["S-pol"]
    return {name: v.reshape(n, n) for name, v in maps.items()}


def _average(g, comp, at):
    """get(): the mean of the two values of a component around a node (E along its axis, H over
    the four around it), real parts."""
    h, axis = (0 if comp[0] == "E" else 1), "xyz".index(comp[1])
    q, i = at[0], list(at[1:])
    spread = [2 if (a == axis) == (h == 0) else 1 for a in range(3)]
    v = g.F[h][axis][(q,) + tuple(slice(c, c + k) for c, k in zip(i, spread))]
    return (v.real if v.is_complex() else v).mean()


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "spectra":
        v = torch.from_numpy(_spectra_samples(case, seed)).to(device)
        tau = torch.tensor([_tau(case, n + 1) for n in range(case["steps"])], dtype=torch.float64, device=device)
        harm = _top(case) - torch.arange(case["bins"], dtype=torch.float64, device=device)
        turn = torch.exp(1j * (2 * math.pi * tau[:, None] * harm))
        out = (v.to(torch.complex128).permute(1, 2, 0).reshape(-1, case["steps"]) @ turn).reshape(case["spectra"], case["probes"], case["bins"])
        return torch.view_as_real(out).cpu().numpy()
    scenes = _scenes(case, seed)
    groups = [scenes] if case["kind"] == "bands" else [[s] for s in scenes]
    names = ("Hz", "Ez") if case["kind"] == "bands" else ("Ez", "Hy")
    out, read, flux = [], [], []
    for group in groups:
        g, s = _grid(group, device), group[0]
        surface = _Surface(g) if s.phaser else None
        at = []
        for q, w in enumerate(group):
            for p, x in enumerate(w.probes):
                node = (q,) + tuple(_node(s, v) - m + 1 for v, m in zip(x, s.MIN))
                at += [(names[p % 2], node)] if case["kind"] == "bands" else [(c, node) for c in names]
        for _ in range(case["steps"]):
            g.half(0)
            g.half(1)
            if surface:
                surface.add(g)
            read += [_average(g, *a) for a in at]
        if case["kind"] == "farfield":
            return _far(surface, case["map"])
        picked = range(0, len(group), max(1, -(-len(group) // 4))) if case["kind"] == "bands" else (0,)
        for q in picked:
            parts = [[v[q, 1:-1, 1:-1, 1:-1].real if v.is_complex() else v[q, 1:-1, 1:-1, 1:-1] for V in g.F for v in V]]
            if s.bloch:
                parts.append([v[q, 1:-1, 1:-1, 1:-1].imag for V in g.F for v in V])
            out.append([v for p in parts for v in p])
        if surface:
            flux.append(surface.flux())
    answer = {"fields": out}
    if read:
        answer["probes"] = torch.stack(read)
    if flux:
        answer["flux"] = flux
    return answer
