"""Host-side mirror of the reference's simulator interface over ``libnbody.so``.

The reference exposes its gravity step as ``INBodySim`` with ``Init``,
``Update`` and ``RenderDebug`` (src/Sim/INBodySim.hpp:19-25), created by
``CreateNBodySim`` and named by ``NBodySimGetName`` (src/Sim/INBodySim.cpp:7-39).
This module offers the same surface in Python, calling the HIP library through
its C ABI (``include/nbody.h``) with ctypes:

* ``ENBodySim`` - the reference's selector (BruteForceCPU, BruteForceGPU,
  BarnesHut); both brute-force entries run the device direct sum.
* ``create_nbody_sim(kind, config=None)`` / ``nbody_sim_get_name(kind)``.
* ``NBodySim.init(particles)`` keeps the caller's record array, like the
  reference keeps a pointer to the caller's ``std::vector<Particle>``, and
  ``NBodySim.update(dt)`` advances one step and writes positions, velocities
  and forces back into it (SimulationState.cpp:52-60).
* ``PARTICLE_DTYPE`` - the reference's 104-byte ``Particle`` record
  (src/Render/Misc/Particle.hpp:8-18), also the ``.nbody`` file record.

The library must be built (``make -C procedural-universe_amd``); there is no
fallback: every call goes to the device code or raises.
"""
from __future__ import annotations

import ctypes
import enum
import os
from typing import Optional

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libnbody.so")

PARTICLE_DTYPE = np.dtype(
    [
        ("position", "<f4", (3,)),
        ("colour", "<f4", (4,)),
        ("original_colour", "<f4", (4,)),
        ("pad_", "<f4"),
        ("velocity", "<f8", (3,)),
        ("forces", "<f8", (3,)),
        ("mass", "<f8"),
    ]
)
assert PARTICLE_DTYPE.itemsize == 104

# nbody_bh_cell (include/nbody.h): one octree cell, 48 bytes.
BH_CELL_DTYPE = np.dtype([
    ("lo", np.float32, 3), ("side", np.float32), ("com", np.float32, 3), ("level", np.uint32),
    ("mass", np.float64), ("first", np.uint32), ("count", np.uint32),
])
assert BH_CELL_DTYPE.itemsize == 48

# nbody_status
OK = 0
STATUS_NAMES = {
    0: "NBODY_OK",
    1: "NBODY_ERR_INVALID_ARG",
    2: "NBODY_ERR_OUT_OF_MEMORY",
    3: "NBODY_ERR_DEVICE",
    4: "NBODY_ERR_NOT_INITIALISED",
    5: "NBODY_ERR_UNSUPPORTED",
    6: "NBODY_ERR_CAPACITY",
    7: "NBODY_ERR_IO",
}

METHOD_DIRECT = 1
# nbody_seeder (EParticleSeeder)
SEEDER_RANDOM = 0
SEEDER_GALAXY = 1
SEEDER_STAR_SYSTEM = 2
METHOD_BARNES_HUT = 2
LAW_R = 0
LAW_P = 1
ROOT_DYNAMIC = 0
ROOT_FIXED = 1
FIELD_POSITION = 1
FIELD_VELOCITY = 2
FIELD_FORCES = 4
FIELD_MASS = 8


class ENBodySim(enum.IntEnum):
    """src/Sim/INBodySim.hpp:11-17."""

    BruteForceCPU = 0
    BruteForceGPU = 1
    BarnesHut = 2
    NumSims = 3


_SIM_NAMES = {
    ENBodySim.BruteForceCPU: "Brute Force CPU",
    ENBodySim.BruteForceGPU: "Brute Force GPU",
    ENBodySim.BarnesHut: "Barnes-Hut",
}


def nbody_sim_get_name(kind) -> str:
    """NBodySimGetName (src/Sim/INBodySim.cpp:29-39)."""
    try:
        return _SIM_NAMES[ENBodySim(kind)]
    except (ValueError, KeyError):
        return "Unknown"


class Config(ctypes.Structure):
    """``nbody_config`` of include/nbody.h."""

    _fields_ = [
        ("method", ctypes.c_int32),
        ("law", ctypes.c_int32),
        ("G", ctypes.c_double),
        ("softening", ctypes.c_double),
        ("scale", ctypes.c_double),
        ("theta", ctypes.c_double),
        ("root_mode", ctypes.c_int32),
        ("root_lo", ctypes.c_float * 3),
        ("root_size", ctypes.c_float),
        ("device", ctypes.c_int32),
        ("tune_i_per_lane", ctypes.c_int32),
        ("tune_block", ctypes.c_int32),
        ("tune_split", ctypes.c_int32),
        ("inject_rows_failures", ctypes.c_int32),
        ("reserved", ctypes.c_int32 * 7),
    ]


class Diag(ctypes.Structure):
    _fields_ = [
        ("kinetic", ctypes.c_double),
        ("potential", ctypes.c_double),
        ("total", ctypes.c_double),
        ("momentum", ctypes.c_double * 3),
        ("angular_momentum", ctypes.c_double * 3),
        ("mass", ctypes.c_double),
    ]

    def as_dict(self):
        return {
            "kinetic": self.kinetic,
            "potential": self.potential,
            "total": self.total,
            "momentum": list(self.momentum),
            "angular_momentum": list(self.angular_momentum),
            "mass": self.mass,
        }


class Timing(ctypes.Structure):
    _fields_ = [
        ("steps", ctypes.c_int32),
        ("force_launches", ctypes.c_int32),
        ("force_ms", ctypes.c_double),
        ("tree_ms", ctypes.c_double),
        ("step_ms", ctypes.c_double),
        ("interactions", ctypes.c_uint64),
        ("i_per_lane", ctypes.c_int32),
        ("block", ctypes.c_int32),
        ("split", ctypes.c_int32),
        ("reserved", ctypes.c_int32 * 5),
    ]


class BHStats(ctypes.Structure):
    _fields_ = [
        ("interactions", ctypes.c_uint64),
        ("outside_root", ctypes.c_uint32),
        ("stack_overflow", ctypes.c_uint32),
        ("list_entries", ctypes.c_uint64),
        ("cells_opened", ctypes.c_uint64),
    ]


class BatchTuning(ctypes.Structure):
    _fields_ = [
        ("i_per_lane", ctypes.c_int32),
        ("block", ctypes.c_int32),
        ("wg_per_cu", ctypes.c_int32),
        ("reserved", ctypes.c_int32 * 5),
        ("ms_per_step", ctypes.c_double),
    ]

    def as_dict(self):
        return {"i_per_lane": self.i_per_lane, "block": self.block, "wg_per_cu": self.wg_per_cu,
                "ms_per_step": self.ms_per_step}


class BatchInfo(ctypes.Structure):
    _fields_ = [
        ("systems", ctypes.c_int32),
        ("work_items", ctypes.c_int32),
        ("particles", ctypes.c_uint64),
        ("interactions_per_step", ctypes.c_uint64),
        ("capacity", ctypes.c_uint64),
        ("free_records", ctypes.c_uint64),
        ("largest_free", ctypes.c_uint64),
        ("tuning", BatchTuning),
    ]


class ServerConfig(ctypes.Structure):
    _fields_ = [
        ("sim", Config),
        ("memory_budget", ctypes.c_uint64),
        ("direct_capacity", ctypes.c_uint64),
        ("bh_threshold", ctypes.c_uint32),
        ("max_active_bh", ctypes.c_int32),
        ("dt", ctypes.c_float),
        ("keep_results", ctypes.c_int32),
        ("bh_steps_ahead", ctypes.c_int32),
        ("inject_alloc_failures", ctypes.c_int32),
        ("bh_no_graph", ctypes.c_int32),
        ("reserved", ctypes.c_int32 * 5),
    ]


class RequestResult(ctypes.Structure):
    _fields_ = [
        ("id", ctypes.c_uint64),
        ("n", ctypes.c_uint32),
        ("steps", ctypes.c_int32),
        ("method", ctypes.c_int32),
        ("pad_", ctypes.c_int32),
        ("arrival", ctypes.c_double),
        ("admitted", ctypes.c_double),
        ("completed", ctypes.c_double),
        ("interactions", ctypes.c_uint64),
    ]


class ServerStats(ctypes.Structure):
    _fields_ = [
        ("submitted", ctypes.c_uint64),
        ("admitted", ctypes.c_uint64),
        ("completed", ctypes.c_uint64),
        ("pending", ctypes.c_uint64),
        ("active_direct", ctypes.c_uint64),
        ("active_bh", ctypes.c_uint64),
        ("idle_handles", ctypes.c_uint64),
        ("memory_used", ctypes.c_uint64),
        ("memory_peak", ctypes.c_uint64),
        ("interactions", ctypes.c_uint64),
        ("ticks", ctypes.c_uint64),
        ("busy_seconds", ctypes.c_double),
        ("alloc_deferrals", ctypes.c_uint64),
    ]

    def as_dict(self):
        return {name: getattr(self, name) for name, _ in self._fields_}


class NBodyError(RuntimeError):
    def __init__(self, func: str, status: int, message: str):
        self.status = status
        super().__init__(f"{func}: {STATUS_NAMES.get(status, status)}: {message}")


_lib = None

_P = ctypes.c_void_p
_F32P = ctypes.POINTER(ctypes.c_float)
_F64P = ctypes.POINTER(ctypes.c_double)

# name -> (restype, argtypes)
_SIGNATURES = {
    "nbody_config_default": (None, [ctypes.POINTER(Config)]),
    "nbody_config_reference": (None, [ctypes.POINTER(Config), ctypes.c_int32]),
    "nbody_create": (ctypes.c_int, [ctypes.POINTER(Config), ctypes.POINTER(_P)]),
    "nbody_destroy": (ctypes.c_int, [_P]),
    "nbody_init": (ctypes.c_int, [_P, _P, ctypes.c_size_t]),
    "nbody_init_soa": (ctypes.c_int, [_P, _F32P, _F32P, _F64P, ctypes.c_size_t]),
    "nbody_step": (ctypes.c_int, [_P, ctypes.c_float, ctypes.c_int32]),
    "nbody_synchronize": (ctypes.c_int, [_P]),
    "nbody_query": (ctypes.c_int, [_P, ctypes.POINTER(ctypes.c_int32)]),
    "nbody_set_graph": (ctypes.c_int, [_P, ctypes.c_int32]),
    "nbody_set_theta": (ctypes.c_int, [_P, ctypes.c_double]),
    "nbody_field_noalloc": (ctypes.c_int, [_P, _F32P, ctypes.c_size_t, _F32P]),
    "nbody_direct_scale": (ctypes.c_int, [ctypes.c_int32, ctypes.c_double, ctypes.c_double, ctypes.c_double, _F32P]),
    "nbody_init_seeded": (ctypes.c_int, [_P, ctypes.c_int32, ctypes.c_uint64, ctypes.c_size_t, ctypes.c_double]),
    "nbody_read": (ctypes.c_int, [_P, _P, ctypes.c_size_t, ctypes.c_uint32]),
    "nbody_read_soa": (ctypes.c_int, [_P, _F32P, _F32P, _F32P, ctypes.c_size_t]),
    "nbody_compute_accelerations": (ctypes.c_int, [_P, _F32P, ctypes.c_size_t]),
    "nbody_size": (ctypes.c_int, [_P, ctypes.POINTER(ctypes.c_size_t)]),
    "nbody_diagnostics": (ctypes.c_int, [_P, ctypes.POINTER(Diag)]),
    "nbody_set_timing": (ctypes.c_int, [_P, ctypes.c_int32]),
    "nbody_get_timing": (ctypes.c_int, [_P, ctypes.POINTER(Timing)]),
    "nbody_bh_stats_get": (ctypes.c_int, [_P, ctypes.POINTER(BHStats)]),
    "nbody_bh_cells": (ctypes.c_int, [_P, ctypes.c_void_p, ctypes.c_size_t, ctypes.POINTER(ctypes.c_size_t)]),
    "nbody_bh_tree_order": (
        ctypes.c_int,
        [_P, ctypes.POINTER(ctypes.c_uint64), ctypes.POINTER(ctypes.c_uint32), ctypes.c_size_t],
    ),
    "nbody_batch_create": (ctypes.c_int, [ctypes.POINTER(Config), ctypes.c_size_t, ctypes.POINTER(_P)]),
    "nbody_batch_destroy": (ctypes.c_int, [_P]),
    "nbody_batch_add": (ctypes.c_int, [_P, _F32P, _F32P, _F64P, ctypes.c_size_t, ctypes.POINTER(ctypes.c_int32)]),
    "nbody_batch_remove": (ctypes.c_int, [_P, ctypes.c_int32]),
    "nbody_batch_step": (ctypes.c_int, [_P, ctypes.c_float, ctypes.c_int32]),
    "nbody_batch_step_sequential": (ctypes.c_int, [_P, ctypes.c_float, ctypes.c_int32, ctypes.c_int32]),
    "nbody_batch_synchronize": (ctypes.c_int, [_P]),
    "nbody_batch_query": (ctypes.c_int, [_P, ctypes.POINTER(ctypes.c_int32)]),
    "nbody_batch_read": (ctypes.c_int, [_P, ctypes.c_int32, _F32P, _F32P, _F32P, ctypes.c_size_t]),
    "nbody_batch_get_info": (ctypes.c_int, [_P, ctypes.POINTER(BatchInfo)]),
    "nbody_batch_set_tuning": (ctypes.c_int, [_P, ctypes.POINTER(BatchTuning)]),
    "nbody_batch_tune": (ctypes.c_int, [_P, ctypes.c_float, ctypes.POINTER(BatchTuning)]),
    "nbody_batch_set_graph": (ctypes.c_int, [_P, ctypes.c_int32]),
    "nbody_batch_get_timing": (ctypes.c_int, [_P, ctypes.POINTER(Timing)]),
    "nbody_init_plummer": (ctypes.c_int, [_P, ctypes.c_uint64, ctypes.c_size_t, ctypes.c_double, ctypes.c_double]),
    "nbody_batch_add_plummer": (
        ctypes.c_int,
        [_P, ctypes.c_uint64, ctypes.c_size_t, ctypes.c_double, ctypes.c_double, ctypes.POINTER(ctypes.c_int32)],
    ),
    "nbody_server_config_default": (None, [ctypes.POINTER(ServerConfig)]),
    "nbody_server_create": (ctypes.c_int, [ctypes.POINTER(ServerConfig), ctypes.POINTER(_P)]),
    "nbody_server_destroy": (ctypes.c_int, [_P]),
    "nbody_server_clock": (ctypes.c_double, [_P]),
    "nbody_server_submit_plummer": (
        ctypes.c_int,
        [_P, ctypes.c_uint64, ctypes.c_size_t, ctypes.c_int32, ctypes.c_double, ctypes.c_double, ctypes.c_double,
         ctypes.POINTER(ctypes.c_uint64)],
    ),
    "nbody_server_tick": (ctypes.c_int, [_P, ctypes.POINTER(ctypes.c_int32)]),
    "nbody_server_poll": (ctypes.c_int, [_P, ctypes.POINTER(RequestResult), ctypes.c_int32, ctypes.POINTER(ctypes.c_int32)]),
    "nbody_server_fetch": (ctypes.c_int, [_P, ctypes.c_uint64, _F32P, _F32P, ctypes.c_size_t]),
    "nbody_server_get_stats": (ctypes.c_int, [_P, ctypes.POINTER(ServerStats)]),
    "nbody_snapshot_count": (ctypes.c_int, [ctypes.c_char_p, ctypes.POINTER(ctypes.c_size_t)]),
    "nbody_snapshot_read": (
        ctypes.c_int, [ctypes.c_char_p, _P, ctypes.c_size_t, ctypes.POINTER(ctypes.c_size_t), ctypes.c_int32]
    ),
    "nbody_snapshot_write": (ctypes.c_int, [ctypes.c_char_p, _P, ctypes.c_size_t]),
    "nbody_method_name": (ctypes.c_char_p, [ctypes.c_int32]),
    "nbody_status_string": (ctypes.c_char_p, [ctypes.c_int]),
    "nbody_last_error": (ctypes.c_char_p, []),
    "nbody_abi_version": (ctypes.c_int32, []),
    "nbody_device_count": (ctypes.c_int32, []),
    "nbody_ic_plummer": (
        ctypes.c_int,
        [ctypes.c_uint64, ctypes.c_size_t, ctypes.c_double, ctypes.c_double, ctypes.c_double, _F32P, _F32P, _F64P],
    ),
    "nbody_ic_disc_bulge": (
        ctypes.c_int,
        [
            ctypes.c_uint64,
            ctypes.c_size_t,
            ctypes.c_double,
            ctypes.c_double,
            ctypes.c_double,
            ctypes.c_double,
            ctypes.c_double,
            ctypes.c_double,
            _F32P,
            _F32P,
            _F64P,
        ],
    ),
    "nbody_field": (ctypes.c_int, [_P, _F32P, ctypes.c_size_t, _F32P]),
    "nbody_ic_disc_encounter": (
        ctypes.c_int,
        [ctypes.c_uint64, ctypes.c_size_t] + [ctypes.c_double] * 6 + [_F32P, _F32P, _F64P],
    ),
    "nbody_ic_uniform": (
        ctypes.c_int,
        [ctypes.c_uint64, ctypes.c_size_t, ctypes.c_double, ctypes.c_double, ctypes.c_double, _F32P, _F32P, _F64P],
    ),
}


def load_library(path: Optional[str] = None) -> ctypes.CDLL:
    """Load libnbody.so (raises OSError when it is not built)."""
    global _lib
    if _lib is not None and path is None:
        return _lib
    p = path or LIB_PATH
    if not os.path.exists(p):
        raise OSError(f"{p} is not built; run `make -C {_HERE}` or __graft_entry__.build()")
    lib = ctypes.CDLL(p)
    for name, (res, args) in _SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    if path is None:
        _lib = lib
    return lib


def _check(func: str, status: int):
    if status != OK:
        msg = load_library().nbody_last_error()
        raise NBodyError(func, status, msg.decode() if msg else "")


def _f32(a):
    return a.ctypes.data_as(_F32P)


def _f64(a):
    return a.ctypes.data_as(_F64P)


def direct_scale(law: int, softening: float, extent: float, max_gm: float) -> dict:
    """The scaled units the direct sum would compute such a system in
    (nbody_direct_scale; host only)."""
    out = np.zeros(4, np.float32)
    _check("nbody_direct_scale", load_library().nbody_direct_scale(int(law), float(softening), float(extent),
                                                                   float(max_gm), _f32(out)))
    return {"inv_len": float(out[0]), "mass_k": float(out[1]), "soft": float(out[2]), "out": float(out[3])}


def device_count() -> int:
    return int(load_library().nbody_device_count())


def default_config(**overrides) -> Config:
    c = Config()
    load_library().nbody_config_default(ctypes.byref(c))
    return _apply(c, overrides)


def reference_config(method: int = METHOD_DIRECT, **overrides) -> Config:
    """The reference's constants (src/Sim/Physics.hpp:9-16, Octree.cpp:5, BarnesHut.cpp:14-19)."""
    c = Config()
    load_library().nbody_config_reference(ctypes.byref(c), int(method))
    return _apply(c, overrides)


def _apply(c: Config, overrides) -> Config:
    for k, v in overrides.items():
        if k == "root_lo":
            for i in range(3):
                c.root_lo[i] = float(v[i])
        else:
            setattr(c, k, v)
    return c


class NBodySim:
    """One device simulation: the INBodySim contract (src/Sim/INBodySim.hpp:19-25)."""

    def __init__(self, config: Config):
        lib = load_library()
        self._lib = lib
        self.config = config
        h = _P()
        _check("nbody_create", lib.nbody_create(ctypes.byref(config), ctypes.byref(h)))
        self._h = h
        self._particles = None
        self.n = 0
        # BruteForceCPU/GPU leave Forces zeroed after Update (BruteForceCPU.cpp:72,
        # Update.csh:35); BarnesHut leaves the last forces (BarnesHut.cpp:75,108).
        self.zero_forces_after_update = config.method == METHOD_DIRECT

    # -- lifetime ---------------------------------------------------------
    def close(self):
        if getattr(self, "_h", None):
            self._lib.nbody_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()

    # -- INBodySim --------------------------------------------------------
    def init(self, particles: np.ndarray):
        """INBodySim::Init: adopt the caller's record array (updated in place by update())."""
        if particles.dtype != PARTICLE_DTYPE or not particles.flags["C_CONTIGUOUS"]:
            raise TypeError("particles must be a C-contiguous array of PARTICLE_DTYPE")
        _check("nbody_init", self._lib.nbody_init(self._h, particles.ctypes.data, particles.size))
        self._particles = particles
        self.n = particles.size

    def update(self, dt: float):
        """INBodySim::Update: one synchronous step, written back into the adopted records."""
        if self._particles is None:
            raise RuntimeError("update() before init()")
        self.step(dt, 1)
        p = self._particles
        _check(
            "nbody_read",
            self._lib.nbody_read(self._h, p.ctypes.data, p.size, FIELD_POSITION | FIELD_VELOCITY | FIELD_FORCES),
        )
        if self.zero_forces_after_update:
            p["forces"] = 0.0

    def render_debug(self, view=None, proj=None):
        """INBodySim::RenderDebug has a do-nothing default (INBodySim.hpp:23)."""
        return None

    # -- structure-of-arrays API ----------------------------------------
    def init_soa(self, pos: np.ndarray, vel: Optional[np.ndarray], mass: np.ndarray):
        pos = np.ascontiguousarray(pos, dtype=np.float32).reshape(-1, 3)
        n = pos.shape[0]
        mass = np.ascontiguousarray(mass, dtype=np.float64).reshape(n)
        velp = None
        if vel is not None:
            vel = np.ascontiguousarray(vel, dtype=np.float32).reshape(n, 3)
            velp = _f32(vel)
        _check("nbody_init_soa", self._lib.nbody_init_soa(self._h, _f32(pos), velp, _f64(mass), n))
        self._particles = None
        self.n = n

    def init_plummer(self, n: int, seed: int, a: float = 1.0, total_mass: float = 1.0):
        """Plummer sphere generated in device memory (same stream as ic_plummer)."""
        _check("nbody_init_plummer", self._lib.nbody_init_plummer(self._h, int(seed), int(n), float(a), float(total_mass)))
        self._particles = None
        self.n = n

    def init_seeded(self, seeder: int, n: int, seed: int = 0, scale: float = 1.0):
        """One of the reference's seeders (SEEDER_RANDOM, SEEDER_GALAXY,
        SEEDER_STAR_SYSTEM) drawn in device memory."""
        _check("nbody_init_seeded", self._lib.nbody_init_seeded(self._h, int(seeder), int(seed), int(n), float(scale)))
        self._particles = None
        self.n = n

    def step(self, dt: float, nsteps: int = 1):
        _check("nbody_step", self._lib.nbody_step(self._h, float(dt), int(nsteps)))

    def synchronize(self):
        _check("nbody_synchronize", self._lib.nbody_synchronize(self._h))

    def query(self) -> bool:
        """True when every enqueued step has completed (does not wait)."""
        done = ctypes.c_int32(0)
        _check("nbody_query", self._lib.nbody_query(self._h, ctypes.byref(done)))
        return bool(done.value)

    def set_graph(self, enable: bool = True):
        """Replay step sequences from captured hipGraphs (bit-identical results)."""
        _check("nbody_set_graph", self._lib.nbody_set_graph(self._h, 1 if enable else 0))

    def set_theta(self, theta: float):
        """Octree::Theta of the live simulation (the reference's BHThetaChanged,
        src/Sim/BarnesHut.cpp:29-31): later steps open cells with it."""
        _check("nbody_set_theta", self._lib.nbody_set_theta(self._h, float(theta)))

    def read_soa(self):
        n = self.n
        pos = np.empty((n, 3), np.float32)
        vel = np.empty((n, 3), np.float32)
        acc = np.empty((n, 3), np.float32)
        _check("nbody_read_soa", self._lib.nbody_read_soa(self._h, _f32(pos), _f32(vel), _f32(acc), n))
        return pos, vel, acc

    def read_particles(self, particles: np.ndarray, fields: int = 7):
        _check("nbody_read", self._lib.nbody_read(self._h, particles.ctypes.data, particles.size, fields))

    def accelerations(self) -> np.ndarray:
        acc = np.empty((self.n, 3), np.float32)
        _check("nbody_compute_accelerations", self._lib.nbody_compute_accelerations(self._h, _f32(acc), self.n))
        return acc

    def field(self, points) -> np.ndarray:
        """Direct-sum acceleration at arbitrary points from the current particles."""
        pts = np.ascontiguousarray(points, dtype=np.float32).reshape(-1, 3)
        out = np.empty_like(pts)
        _check("nbody_field", self._lib.nbody_field(self._h, _f32(pts), pts.shape[0], _f32(out)))
        return out

    def diagnostics(self) -> dict:
        d = Diag()
        _check("nbody_diagnostics", self._lib.nbody_diagnostics(self._h, ctypes.byref(d)))
        return d.as_dict()

    def bh_stats(self) -> dict:
        st = BHStats()
        _check("nbody_bh_stats_get", self._lib.nbody_bh_stats_get(self._h, ctypes.byref(st)))
        return {"interactions": int(st.interactions), "outside_root": int(st.outside_root),
                "stack_overflow": int(st.stack_overflow), "list_entries": int(st.list_entries),
                "cells_opened": int(st.cells_opened)}

    def bh_tree_order(self):
        """Sorted Morton keys and particle order of the last Barnes-Hut tree build."""
        keys = np.empty(self.n, np.uint64)
        order = np.empty(self.n, np.uint32)
        _check(
            "nbody_bh_tree_order",
            self._lib.nbody_bh_tree_order(
                self._h, keys.ctypes.data_as(ctypes.POINTER(ctypes.c_uint64)),
                order.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), self.n
            ),
        )
        return keys, order

    def bh_cells(self) -> np.ndarray:
        """Octree cells of the last Barnes-Hut tree build (structured array of
        lo[3], side, com[3], level, mass, first, count), depth-first."""
        count = ctypes.c_size_t(0)
        _check("nbody_bh_cells", self._lib.nbody_bh_cells(self._h, None, 0, ctypes.byref(count)))
        out = np.zeros(count.value, dtype=BH_CELL_DTYPE)
        got = ctypes.c_size_t(0)
        _check("nbody_bh_cells", self._lib.nbody_bh_cells(self._h, out.ctypes.data_as(ctypes.c_void_p),
                                                          count.value, ctypes.byref(got)))
        return out

    def set_timing(self, enable: bool = True):
        _check("nbody_set_timing", self._lib.nbody_set_timing(self._h, 1 if enable else 0))

    def timing(self) -> Timing:
        t = Timing()
        _check("nbody_get_timing", self._lib.nbody_get_timing(self._h, ctypes.byref(t)))
        return t


class Batch:
    """Many independent systems advanced together (include/nbody.h, nbody_batch_*)."""

    def __init__(self, config: Config, capacity: int):
        lib = load_library()
        self._lib = lib
        self.config = config
        h = _P()
        _check("nbody_batch_create", lib.nbody_batch_create(ctypes.byref(config), int(capacity), ctypes.byref(h)))
        self._h = h
        self.sizes = {}

    def close(self):
        if getattr(self, "_h", None):
            self._lib.nbody_batch_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()

    def add(self, pos, vel, mass) -> int:
        pos = np.ascontiguousarray(pos, dtype=np.float32).reshape(-1, 3)
        n = pos.shape[0]
        mass = np.ascontiguousarray(mass, dtype=np.float64).reshape(n)
        velp = None
        if vel is not None:
            vel = np.ascontiguousarray(vel, dtype=np.float32).reshape(n, 3)
            velp = _f32(vel)
        sid = ctypes.c_int32()
        _check("nbody_batch_add", self._lib.nbody_batch_add(self._h, _f32(pos), velp, _f64(mass), n, ctypes.byref(sid)))
        self.sizes[sid.value] = n
        return sid.value

    def add_plummer(self, n: int, seed: int, a: float = 1.0, total_mass: float = 1.0) -> int:
        sid = ctypes.c_int32()
        _check(
            "nbody_batch_add_plummer",
            self._lib.nbody_batch_add_plummer(self._h, int(seed), int(n), float(a), float(total_mass), ctypes.byref(sid)),
        )
        self.sizes[sid.value] = n
        return sid.value

    def remove(self, sid: int):
        _check("nbody_batch_remove", self._lib.nbody_batch_remove(self._h, int(sid)))
        self.sizes.pop(sid, None)

    def step(self, dt: float, nsteps: int = 1):
        _check("nbody_batch_step", self._lib.nbody_batch_step(self._h, float(dt), int(nsteps)))

    def step_sequential(self, dt: float, nsteps: int = 1, split_small: bool = False):
        _check(
            "nbody_batch_step_sequential",
            self._lib.nbody_batch_step_sequential(self._h, float(dt), int(nsteps), 1 if split_small else 0),
        )

    def synchronize(self):
        _check("nbody_batch_synchronize", self._lib.nbody_batch_synchronize(self._h))

    def query(self) -> bool:
        """True when every enqueued step has completed (does not wait)."""
        done = ctypes.c_int32(0)
        _check("nbody_batch_query", self._lib.nbody_batch_query(self._h, ctypes.byref(done)))
        return bool(done.value)

    def read(self, sid: int):
        n = self.sizes[sid]
        pos = np.empty((n, 3), np.float32)
        vel = np.empty((n, 3), np.float32)
        acc = np.empty((n, 3), np.float32)
        _check("nbody_batch_read", self._lib.nbody_batch_read(self._h, int(sid), _f32(pos), _f32(vel), _f32(acc), n))
        return pos, vel, acc

    def info(self) -> BatchInfo:
        inf = BatchInfo()
        _check("nbody_batch_get_info", self._lib.nbody_batch_get_info(self._h, ctypes.byref(inf)))
        return inf

    def set_tuning(self, i_per_lane: int, block: int, wg_per_cu: int):
        t = BatchTuning(i_per_lane, block, wg_per_cu)
        _check("nbody_batch_set_tuning", self._lib.nbody_batch_set_tuning(self._h, ctypes.byref(t)))

    def tune(self, dt: float) -> dict:
        t = BatchTuning()
        _check("nbody_batch_tune", self._lib.nbody_batch_tune(self._h, float(dt), ctypes.byref(t)))
        return t.as_dict()

    def set_graph(self, enable: bool):
        _check("nbody_batch_set_graph", self._lib.nbody_batch_set_graph(self._h, 1 if enable else 0))

    def timing(self) -> Timing:
        t = Timing()
        _check("nbody_batch_get_timing", self._lib.nbody_batch_get_timing(self._h, ctypes.byref(t)))
        return t


def server_config(**overrides) -> ServerConfig:
    c = ServerConfig()
    load_library().nbody_server_config_default(ctypes.byref(c))
    for k, v in overrides.items():
        if k == "sim":
            c.sim = v
        elif hasattr(c.sim, k) and not hasattr(c, k):
            setattr(c.sim, k, v)
        else:
            setattr(c, k, v)
    return c


class Server:
    """Continuous-batching request server (include/nbody.h, nbody_server_*)."""

    def __init__(self, config: ServerConfig):
        lib = load_library()
        self._lib = lib
        self.config = config
        h = _P()
        _check("nbody_server_create", lib.nbody_server_create(ctypes.byref(config), ctypes.byref(h)))
        self._h = h

    def close(self):
        if getattr(self, "_h", None):
            self._lib.nbody_server_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()

    def clock(self) -> float:
        return float(self._lib.nbody_server_clock(self._h))

    def submit_plummer(self, n: int, steps: int, seed: int, a: float = 1.0, total_mass: float = 1.0,
                       arrival: float = float("nan")) -> int:
        rid = ctypes.c_uint64()
        _check(
            "nbody_server_submit_plummer",
            self._lib.nbody_server_submit_plummer(self._h, int(seed), int(n), int(steps), float(a), float(total_mass),
                                                  float(arrival), ctypes.byref(rid)),
        )
        return rid.value

    def tick(self) -> int:
        c = ctypes.c_int32()
        _check("nbody_server_tick", self._lib.nbody_server_tick(self._h, ctypes.byref(c)))
        return c.value

    def poll(self, max_results: int = 4096):
        buf = (RequestResult * max_results)()
        c = ctypes.c_int32()
        _check("nbody_server_poll", self._lib.nbody_server_poll(self._h, buf, max_results, ctypes.byref(c)))
        return [
            {"id": r.id, "n": r.n, "steps": r.steps, "method": r.method, "arrival": r.arrival, "admitted": r.admitted,
             "completed": r.completed, "interactions": r.interactions}
            for r in buf[: c.value]
        ]

    def fetch(self, rid: int, n: int):
        pos = np.empty((n, 3), np.float32)
        vel = np.empty((n, 3), np.float32)
        _check("nbody_server_fetch", self._lib.nbody_server_fetch(self._h, int(rid), _f32(pos), _f32(vel), n))
        return pos, vel

    def stats(self) -> dict:
        st = ServerStats()
        _check("nbody_server_get_stats", self._lib.nbody_server_get_stats(self._h, ctypes.byref(st)))
        return st.as_dict()


def create_nbody_sim(kind, config: Optional[Config] = None) -> NBodySim:
    """CreateNBodySim (src/Sim/INBodySim.cpp:7-27): reference constants unless a config is given."""
    kind = ENBodySim(kind)
    if kind == ENBodySim.NumSims:
        raise ValueError("NumSims is not a simulator")
    method = METHOD_BARNES_HUT if kind == ENBodySim.BarnesHut else METHOD_DIRECT
    if config is None:
        config = reference_config(method)
    else:
        config.method = method
    return NBodySim(config)


# -- initial conditions ----------------------------------------------------
def _ic_out(n):
    return np.empty((n, 3), np.float32), np.empty((n, 3), np.float32), np.empty(n, np.float64)


def ic_plummer(n: int, seed: int, a: float = 1.0, total_mass: float = 1.0, G: float = 1.0):
    pos, vel, mass = _ic_out(n)
    _check(
        "nbody_ic_plummer",
        load_library().nbody_ic_plummer(seed, n, a, total_mass, G, _f32(pos), _f32(vel), _f64(mass)),
    )
    return pos, vel, mass


def ic_disc_bulge(
    n: int,
    seed: int,
    Rd: float = 3.0,
    z0: float = 0.3,
    bulge_fraction: float = 0.2,
    ab: float = 0.6,
    total_mass: float = 1.0,
    G: float = 1.0,
):
    pos, vel, mass = _ic_out(n)
    _check(
        "nbody_ic_disc_bulge",
        load_library().nbody_ic_disc_bulge(
            seed, n, Rd, z0, bulge_fraction, ab, total_mass, G, _f32(pos), _f32(vel), _f64(mass)
        ),
    )
    return pos, vel, mass


def ic_disc_encounter(n: int, seed: int, Rd: float = 3.0, z0: float = 0.3, separation: float = 40.0,
                      pericentre: float = 5.0, tilt_deg: float = 30.0, G: float = 1.0):
    pos, vel, mass = _ic_out(n)
    _check(
        "nbody_ic_disc_encounter",
        load_library().nbody_ic_disc_encounter(
            seed, n, Rd, z0, separation, pericentre, tilt_deg, G, _f32(pos), _f32(vel), _f64(mass)
        ),
    )
    return pos, vel, mass


def ic_uniform(n: int, seed: int, half: float = 500.0, mass_lo: float = 1e20, mass_hi: float = 1e30):
    pos, vel, mass = _ic_out(n)
    _check(
        "nbody_ic_uniform",
        load_library().nbody_ic_uniform(seed, n, half, mass_lo, mass_hi, _f32(pos), _f32(vel), _f64(mass)),
    )
    return pos, vel, mass


def batch_galaxies(count: int, seed: int, n_lo: int = 1024, n_hi: int = 65536):
    """The mixed-size galaxy set: sizes log-uniform in [n_lo, n_hi], each a Plummer
    sphere or an exponential disc with probability 1/2, seeded per galaxy."""
    rng = np.random.default_rng(seed)
    sizes = np.rint(n_lo * (n_hi / n_lo) ** rng.random(count)).astype(np.int64)
    kinds = rng.random(count) < 0.5
    out = []
    for k in range(count):
        n = int(sizes[k])
        if kinds[k]:
            p, v, m = ic_plummer(n, seed * 100003 + k)
        else:
            p, v, m = ic_disc_bulge(n, seed * 100003 + k, bulge_fraction=0.0)
        out.append((p, v, m))
    return out


def read_snapshot(path: str, recentre: bool = True) -> np.ndarray:
    """A .nbody file as PARTICLE_DTYPE records (SimulationState.cpp:229-277)."""
    lib = load_library()
    n = ctypes.c_size_t()
    _check("nbody_snapshot_count", lib.nbody_snapshot_count(os.fsencode(path), ctypes.byref(n)))
    out = np.zeros(n.value, PARTICLE_DTYPE)
    got = ctypes.c_size_t()
    _check(
        "nbody_snapshot_read",
        lib.nbody_snapshot_read(os.fsencode(path), out.ctypes.data, out.size, ctypes.byref(got), 1 if recentre else 0),
    )
    return out


def write_snapshot(path: str, particles: np.ndarray):
    """Write PARTICLE_DTYPE records as a .nbody file (SimulationState.cpp:317-331)."""
    if particles.dtype != PARTICLE_DTYPE or not particles.flags["C_CONTIGUOUS"]:
        raise TypeError("particles must be a C-contiguous array of PARTICLE_DTYPE")
    _check("nbody_snapshot_write", load_library().nbody_snapshot_write(os.fsencode(path), particles.ctypes.data,
                                                                         particles.size))


def particles_from_soa(pos, vel, mass) -> np.ndarray:
    """Pack SoA arrays into reference-layout records (colours zero)."""
    n = len(mass)
    p = np.zeros(n, PARTICLE_DTYPE)
    p["position"] = pos
    p["velocity"] = vel
    p["mass"] = mass
    return p
