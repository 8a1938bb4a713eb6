"""Python plumbing over the hemepure_amd C ABI (include/hemepure_amd.h).

The library is the product: HIP kernels for gfx950 plus the host-side lattice
builder behind an ``extern "C"`` boundary.  This module only binds it with
ctypes for tests and benchmarks; it never computes anything itself and raises
if the native library is missing.
"""
from __future__ import annotations

import ctypes as C
from pathlib import Path

import numpy as np

PKG = Path(__file__).resolve().parent
LIB_PATH = PKG / "libhemepure_amd.so"

# Constants of include/hemepure_amd.h.
LINK_NONE, LINK_WALL, LINK_INLET, LINK_OUTLET = 0, 1, 2, 3
KERNEL_LBGK, KERNEL_TRT, KERNEL_LES = 0, 1, 2
WALL_SBB, WALL_BFL, WALL_GZS = 0, 1, 2
IOLET_NASH, IOLET_LADD = 0, 1
COSINE, PARABOLIC, FILEVEL, WK2, WK3, FILEPRES, WOMERSLEY = 0, 1, 2, 3, 4, 5, 6
FP64, FP32_SHIFTED = 0, 1
ORDER_AUTO, ORDER_TILE, ORDER_LAYER = 0, 1, 2
STEP_PROPERTIES = 1
(FIELD_PRESSURE, FIELD_VELOCITY, FIELD_SHEAR_STRESS, FIELD_VON_MISES_STRESS, FIELD_SHEAR_RATE,
 FIELD_STRESS_TENSOR, FIELD_TRACTION, FIELD_TANGENTIAL_PROJECTION_TRACTION, FIELD_NORMAL_PROJECTION_TRACTION,
 FIELD_WALL_EXTENSION, FIELD_DISTRIBUTIONS, FIELD_MPI_RANK) = range(12)
(SELECT_WHOLE, SELECT_SURFACE, SELECT_INLET, SELECT_OUTLET, SELECT_PLANE, SELECT_SPHERE, SELECT_LINE,
 SELECT_SURFACE_POINT, SELECT_SURFACE_SPHERE) = range(9)
Q = 19
NO_VALUE = np.finfo(np.float64).max


class HlbError(RuntimeError):
    def __init__(self, code: int, msg: str):
        super().__init__(f"hemepure_amd error {code}: {msg}")
        self.code = code


class GeometryView(C.Structure):
    _fields_ = [
        ("blocks", C.c_int32 * 3),
        ("block_size", C.c_int32),
        ("n_sites", C.c_int64),
        ("coords", C.POINTER(C.c_int32)),
        ("link_type", C.POINTER(C.c_uint8)),
        ("link_iolet", C.POINTER(C.c_int32)),
        ("link_dist", C.POINTER(C.c_float)),
        ("normal_avail", C.POINTER(C.c_uint8)),
        ("normal", C.POINTER(C.c_float)),
    ]


class IoletDesc(C.Structure):
    _fields_ = [
        ("kind", C.c_int32),
        ("warmup", C.c_int32),
        ("position", C.c_double * 3),
        ("normal", C.c_double * 3),
        ("radius", C.c_double),
        ("density_mean", C.c_double),
        ("density_amp", C.c_double),
        ("phase", C.c_double),
        ("period", C.c_double),
        ("max_speed", C.c_double),
        ("table", C.POINTER(C.c_double)),
        ("table_len", C.c_int64),
        ("density_min", C.c_double),
        ("pressure_gradient_amplitude", C.c_double),
        ("womersley_number", C.c_double),
        ("area", C.c_double),
        ("resistance", C.c_double),
        ("r_c", C.c_double),
        ("r_p", C.c_double),
        ("capacitance", C.c_double),
    ]


class Params(C.Structure):
    _fields_ = [
        ("kernel", C.c_int32),
        ("wall_bc", C.c_int32),
        ("inlet_bc", C.c_int32),
        ("outlet_bc", C.c_int32),
        ("precision", C.c_int32),
        ("slab_order", C.c_int32),
        ("tau", C.c_double),
        ("trt_lambda", C.c_double),
    ]


class IoletGeom(C.Structure):
    _fields_ = [
        ("is_inlet", C.c_int32),
        ("id", C.c_int32),
        ("position", C.c_double * 3),
        ("normal", C.c_double * 3),
        ("radius", C.c_double),
    ]


class Request(C.Structure):
    _fields_ = [
        ("geom", C.POINTER(GeometryView)),
        ("params", Params),
        ("inlets", C.POINTER(IoletDesc)),
        ("n_inlets", C.c_int32),
        ("pad0_", C.c_int32),
        ("outlets", C.POINTER(IoletDesc)),
        ("n_outlets", C.c_int32),
        ("pad1_", C.c_int32),
        ("max_steps", C.c_int64),
        ("period", C.c_int64),
        ("tolerance", C.c_double),
        ("rho0", C.c_double),
    ]


class RequestStatus(C.Structure):
    _fields_ = [
        ("state", C.c_int32),
        ("cycles", C.c_int32),
        ("steps", C.c_int64),
        ("sites", C.c_int64),
        ("device_bytes", C.c_int64),
        ("delta", C.c_double),
        ("t_submit", C.c_double),
        ("t_admit", C.c_double),
        ("t_done", C.c_double),
    ]


class XtrSpec(C.Structure):
    _fields_ = [("fields", C.POINTER(C.c_int32)), ("names", C.POINTER(C.c_char_p)), ("n_fields", C.c_int32),
                ("selector", C.c_int32),
                ("voxel_size", C.c_double), ("time_step", C.c_double), ("origin", C.c_double * 3),
                ("point", C.c_double * 3), ("normal", C.c_double * 3), ("radius", C.c_double),
                ("point2", C.c_double * 3)]


REQ_QUEUED, REQ_RUNNING, REQ_CONVERGED, REQ_DONE, REQ_FAILED = 0, 1, 2, 3, 4
SERVE_BATCHED, SERVE_PLAIN = 0, 1

_lib = None

_SIGS = {
    "hlb_last_error": (C.c_char_p, []),
    "hlb_create": (C.c_int, [C.POINTER(GeometryView), C.POINTER(Params), C.POINTER(IoletDesc), C.c_int,
                             C.POINTER(IoletDesc), C.c_int, C.POINTER(C.c_void_p)]),
    "hlb_destroy": (None, [C.c_void_p]),
    "hlb_init_equilibrium": (C.c_int, [C.c_void_p, C.c_double, C.c_int64]),
    "hlb_upload_f": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int64]),
    "hlb_step": (C.c_int, [C.c_void_p, C.c_int64, C.c_uint32]),
    "hlb_step_timed": (C.c_int, [C.c_void_p, C.c_int64, C.c_uint32, C.POINTER(C.c_double)]),
    "hlb_synchronize": (C.c_int, [C.c_void_p]),
    "hlb_download_f": (C.c_int, [C.c_void_p, C.c_void_p]),
    "hlb_get_fields": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]),
    "hlb_timestep": (C.c_int64, [C.c_void_p]),
    "hlb_stability": (C.c_int, [C.c_void_p, C.POINTER(C.c_int)]),
    "hlb_iolet_state": (C.c_int, [C.c_void_p, C.c_int, C.c_int, C.c_void_p]),
    "hlb_monitor": (C.c_int, [C.c_void_p, C.c_void_p]),
    "hlb_monitor_noalloc": (C.c_int, [C.c_void_p, C.c_void_p]),
    "hlb_noalloc_scratch_bytes": (C.c_int64, []),
    "hlb_set_variant": (C.c_int, [C.c_void_p, C.c_int]),
    "hlb_set_graphs": (C.c_int, [C.c_void_p, C.c_int]),
    "hlb_captured_graphs": (C.c_int, [C.c_void_p]),
    "hlb_variant": (C.c_int, [C.c_void_p]),
    "hlb_autotune": (C.c_int, [C.c_void_p, C.c_int64, C.POINTER(C.c_int), C.POINTER(C.c_double)]),
    "hlb_set_params": (C.c_int, [C.c_void_p, C.POINTER(Params)]),
    "hlb_set_sponge": (C.c_int, [C.c_void_p, C.c_double, C.c_double, C.c_int64]),
    "hlb_get_params": (C.c_int, [C.c_void_p, C.POINTER(Params)]),
    "hlb_set_iolets": (C.c_int, [C.c_void_p, C.POINTER(IoletDesc), C.c_int, C.POINTER(IoletDesc), C.c_int]),
    "hlb_device_bytes": (C.c_int64, [C.c_void_p]),
    "hlb_server_create": (C.c_int, [C.c_int64, C.c_int64, C.POINTER(C.c_void_p)]),
    "hlb_server_destroy": (None, [C.c_void_p]),
    "hlb_server_set_mode": (C.c_int, [C.c_void_p, C.c_int]),
    "hlb_server_submit": (C.c_int, [C.c_void_p, C.POINTER(Request), C.POINTER(C.c_int64)]),
    "hlb_server_advance": (C.c_int, [C.c_void_p, C.POINTER(C.c_int), C.POINTER(C.c_int)]),
    "hlb_server_status": (C.c_int, [C.c_void_p, C.c_int64, C.POINTER(RequestStatus)]),
    "hlb_server_fields": (C.c_int, [C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p]),
    "hlb_server_release": (C.c_int, [C.c_void_p, C.c_int64]),
    "hlb_server_site_steps": (C.c_int64, [C.c_void_p]),
    "hlb_server_bytes_in_use": (C.c_int64, [C.c_void_p]),
    "hlb_batch_create": (C.c_int, [C.POINTER(C.c_void_p)]),
    "hlb_batch_destroy": (None, [C.c_void_p]),
    "hlb_batch_add": (C.c_int, [C.c_void_p, C.c_void_p]),
    "hlb_batch_remove": (C.c_int, [C.c_void_p, C.c_void_p]),
    "hlb_batch_size": (C.c_int, [C.c_void_p]),
    "hlb_batch_sites": (C.c_int64, [C.c_void_p]),
    "hlb_batch_step": (C.c_int, [C.c_void_p, C.c_int64, C.c_uint32]),
    "hlb_batch_step_timed": (C.c_int, [C.c_void_p, C.c_int64, C.c_uint32, C.POINTER(C.c_double)]),
    "hlb_batch_set_graphs": (C.c_int, [C.c_void_p, C.c_int]),
    "hlb_batch_captured_graphs": (C.c_int, [C.c_void_p]),
    "hlb_batch_set_variant": (C.c_int, [C.c_void_p, C.c_int]),
    "hlb_batch_variant": (C.c_int, [C.c_void_p]),
    "hlb_batch_autotune": (C.c_int, [C.c_void_p, C.c_int64, C.POINTER(C.c_int), C.POINTER(C.c_double)]),
    "hlb_xtr_open": (C.c_int, [C.c_void_p, C.c_char_p, C.POINTER(XtrSpec), C.POINTER(C.c_void_p)]),
    "hlb_xtr_capture": (C.c_int, [C.c_void_p]),
    "hlb_xtr_write": (C.c_int, [C.c_void_p, C.POINTER(C.c_int64)]),
    "hlb_xtr_write_fields": (C.c_int, [C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p,
                                       C.c_void_p, C.c_void_p]),
    "hlb_get_stress": (C.c_int, [C.c_void_p] + [C.c_void_p] * 6),
    "hlb_get_stress_rows": (C.c_int, [C.c_void_p, C.c_void_p]),
    "hlb_xtr_site_count": (C.c_int64, [C.c_void_p]),
    "hlb_xtr_close": (None, [C.c_void_p]),
    "hlb_checkpoint_read": (C.c_int, [C.c_void_p, C.c_char_p, C.c_int64, C.POINTER(C.c_int64),
                                      C.c_void_p]),
    "hlb_iolet_file_table": (C.c_int, [C.c_char_p, C.c_int, C.c_int64, C.c_double, C.c_double, C.c_void_p,
                                       C.c_int64, C.POINTER(C.c_double)]),
    "hlb_site_count": (C.c_int64, [C.c_void_p]),
    "hlb_class_counts": (C.c_int, [C.c_void_p, C.c_void_p]),
    "hlb_site_coords": (C.c_int, [C.c_void_p, C.c_void_p]),
    "hlb_neighbour_tables": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "hlb_site_masks": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]),
    "hlb_wall_geometry": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "hlb_geom_cylinder": (C.c_int, [C.c_double, C.c_int32, C.c_int32, C.POINTER(C.c_void_p)]),
    "hlb_geom_ybifurcation": (C.c_int, [C.c_double, C.c_double, C.c_double, C.c_double, C.c_double,
                                        C.c_double, C.c_uint64, C.POINTER(C.c_void_p)]),
    "hlb_geom_stenosed_pipe": (C.c_int, [C.c_double, C.c_int32, C.c_double, C.c_double,
                                         C.POINTER(C.c_void_p)]),
    "hlb_geom_vessel_tree": (C.c_int, [C.c_uint64, C.c_int32, C.c_double, C.c_double, C.c_double, C.c_double,
                                       C.c_double, C.POINTER(C.c_int32), C.c_int32, C.POINTER(C.c_void_p)]),
    "hlb_geom_view": (C.c_int, [C.c_void_p, C.POINTER(GeometryView)]),
    "hlb_geom_read_gmy": (C.c_int, [C.c_char_p, C.c_int, C.POINTER(C.c_void_p)]),
    "hlb_geom_iolets": (C.c_int, [C.c_void_p, C.POINTER(IoletGeom), C.c_int]),
    "hlb_geom_free": (None, [C.c_void_p]),
}


def lib() -> C.CDLL:
    """Loads the native library; raises if it has not been built."""
    global _lib
    if _lib is None:
        if not LIB_PATH.exists():
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with `python -m hemepure_amd.build` "
                "(there is no fallback implementation)")
        handle = C.CDLL(str(LIB_PATH))
        for name, (res, args) in _SIGS.items():
            fn = getattr(handle, name)
            fn.restype = res
            fn.argtypes = args
        _lib = handle
    return _lib


def _check(rc: int) -> int:
    if rc < 0:
        raise HlbError(rc, lib().hlb_last_error().decode())
    return rc


def _ptr(a: np.ndarray) -> C.c_void_p:
    return C.c_void_p(a.ctypes.data)


class Geometry:
    """Per-site geometry records: what GeometryReader yields from a .gmy file."""

    def __init__(self, blocks, coords, link_type, link_iolet, link_dist, normal_avail, normal,
                 iolets=None, block_size=8, _owner=None):
        self.blocks = tuple(int(b) for b in blocks)
        self.block_size = int(block_size)
        self.coords = np.ascontiguousarray(coords, dtype=np.int32).reshape(-1, 3)
        n = self.coords.shape[0]
        self.link_type = np.ascontiguousarray(link_type, dtype=np.uint8).reshape(n, 18)
        self.link_iolet = np.ascontiguousarray(link_iolet, dtype=np.int32).reshape(n, 18)
        self.link_dist = np.ascontiguousarray(link_dist, dtype=np.float32).reshape(n, 18)
        self.normal_avail = np.ascontiguousarray(normal_avail, dtype=np.uint8).reshape(n)
        self.normal = np.ascontiguousarray(normal, dtype=np.float32).reshape(n, 3)
        self.iolets = list(iolets or [])
        self._owner = _owner

    @property
    def n_sites(self) -> int:
        return int(self.coords.shape[0])

    def view(self) -> GeometryView:
        v = GeometryView()
        v.blocks[:] = self.blocks
        v.block_size = self.block_size
        v.n_sites = self.n_sites
        v.coords = self.coords.ctypes.data_as(C.POINTER(C.c_int32))
        v.link_type = self.link_type.ctypes.data_as(C.POINTER(C.c_uint8))
        v.link_iolet = self.link_iolet.ctypes.data_as(C.POINTER(C.c_int32))
        v.link_dist = self.link_dist.ctypes.data_as(C.POINTER(C.c_float))
        v.normal_avail = self.normal_avail.ctypes.data_as(C.POINTER(C.c_uint8))
        v.normal = self.normal.ctypes.data_as(C.POINTER(C.c_float))
        return v

    @classmethod
    def _from_native(cls, gptr: C.c_void_p) -> "Geometry":
        L = lib()
        v = GeometryView()
        try:
            _check(L.hlb_geom_view(gptr, C.byref(v)))
            n = v.n_sites

            def arr(p, count, dt):
                if count == 0:
                    return np.zeros(0, dtype=dt)
                return np.ctypeslib.as_array(p, shape=(count,)).astype(dt, copy=True)

            nio = _check(L.hlb_geom_iolets(gptr, None, 0))
            ios = (IoletGeom * max(nio, 1))()
            L.hlb_geom_iolets(gptr, ios, nio)
            iolets = [dict(is_inlet=bool(ios[i].is_inlet), id=int(ios[i].id),
                           position=tuple(ios[i].position), normal=tuple(ios[i].normal),
                           radius=float(ios[i].radius)) for i in range(nio)]
            return cls(tuple(v.blocks), arr(v.coords, 3 * n, np.int32), arr(v.link_type, 18 * n, np.uint8),
                       arr(v.link_iolet, 18 * n, np.int32), arr(v.link_dist, 18 * n, np.float32),
                       arr(v.normal_avail, n, np.uint8), arr(v.normal, 3 * n, np.float32), iolets,
                       v.block_size)
        finally:
            L.hlb_geom_free(gptr)

    @classmethod
    def read_gmy(cls, path, gmy_plus: bool = False) -> "Geometry":
        """A HemeLB .gmy (version 4) file; .gmy+ with gmy_plus.  The file holds
        no iolet positions: give them from the case's XML."""
        g = C.c_void_p()
        _check(lib().hlb_geom_read_gmy(str(path).encode(), 1 if gmy_plus else 0, C.byref(g)))
        return cls._from_native(g)

    @classmethod
    def cylinder(cls, radius: float, length: int, box_xy: int) -> "Geometry":
        g = C.c_void_p()
        _check(lib().hlb_geom_cylinder(radius, length, box_xy, C.byref(g)))
        return cls._from_native(g)

    @classmethod
    def ybifurcation(cls, rp=24.0, lp=200.0, rd=19.0, ld=160.0, angle_deg=30.0, jitter=0.03,
                     seed=2026) -> "Geometry":
        g = C.c_void_p()
        _check(lib().hlb_geom_ybifurcation(rp, lp, rd, ld, angle_deg, jitter, seed, C.byref(g)))
        return cls._from_native(g)

    @classmethod
    def stenosed_pipe(cls, radius: float, length: int, area_reduction: float, width: float) -> "Geometry":
        g = C.c_void_p()
        _check(lib().hlb_geom_stenosed_pipe(radius, length, area_reduction, width, C.byref(g)))
        return cls._from_native(g)

    @classmethod
    def vessel_tree(cls, seed=2026, generations=6, root_radius=40.0, taper=0.79, length_factor=6.0,
                    angle_min=20.0, angle_max=45.0, box=(1024, 1024, 768), threads=0) -> "Geometry":
        g = C.c_void_p()
        b = (C.c_int32 * 3)(*box)
        _check(lib().hlb_geom_vessel_tree(int(seed), int(generations), root_radius, taper, length_factor, angle_min,
                                          angle_max, b, int(threads), C.byref(g)))
        return cls._from_native(g)

    def inlets(self):
        return sorted((i for i in self.iolets if i["is_inlet"]), key=lambda i: i["id"])

    def outlets(self):
        return sorted((i for i in self.iolets if not i["is_inlet"]), key=lambda i: i["id"])


def iolet_desc(kind: int, position, normal, radius=0.0, density_mean=1.0, density_amp=0.0, phase=0.0,
               period=1.0, warmup=0, max_speed=0.0, table=None, area=1.0, resistance=1.0, r_c=1.0,
               r_p=1.0, capacitance=1.0, density_min=1.0, pressure_gradient_amplitude=0.0,
               womersley_number=0.0) -> IoletDesc:
    d = IoletDesc()
    d.kind = kind
    d.warmup = warmup
    d.position[:] = tuple(position)
    d.normal[:] = tuple(normal)
    d.radius = radius
    d.density_mean = density_mean
    d.density_amp = density_amp
    d.phase = phase
    d.period = period
    d.max_speed = max_speed
    if table is not None:
        t = np.ascontiguousarray(table, dtype=np.float64)
        d._table_keepalive = t
        d.table = t.ctypes.data_as(C.POINTER(C.c_double))
        d.table_len = t.size
    d.density_min = density_min
    d.pressure_gradient_amplitude = pressure_gradient_amplitude
    d.womersley_number = womersley_number
    d.area = area
    d.resistance = resistance
    d.r_c = r_c
    d.r_p = r_p
    d.capacitance = capacitance
    return d


def iolet_file_table(path, velocity: bool, total_steps: int, time_step: float, voxel_size: float):
    """InOutLetFile / InOutLetFileVelocity::CalculateTable: (table, density_min)
    with table[0..total_steps] in lattice density or lattice speed."""
    out = np.empty(int(total_steps) + 1, np.float64)
    dmin = C.c_double()
    _check(lib().hlb_iolet_file_table(str(path).encode(), 1 if velocity else 0, int(total_steps), time_step,
                                      voxel_size, _ptr(out), out.size, C.byref(dmin)))
    return out, float(dmin.value)


# Launch variants hlb_set_variant / hlb_autotune accept: 54 tile shapes x
# orders x occupancy levels, with cached or non-temporal row stores; the
# FP32-shifted form also with two slabs per wavefront.
FP64_VARIANTS = 108
FP32_VARIANTS = 216


def variant_count(precision: int) -> int:
    return FP32_VARIANTS if precision == FP32_SHIFTED else FP64_VARIANTS


def params(kernel=KERNEL_LBGK, wall_bc=WALL_SBB, inlet_bc=IOLET_NASH, outlet_bc=IOLET_NASH, tau=0.8,
           trt_lambda=3.0 / 16.0, precision=FP64, slab_order=ORDER_AUTO) -> Params:
    p = Params()
    p.kernel, p.wall_bc, p.inlet_bc, p.outlet_bc = kernel, wall_bc, inlet_bc, outlet_bc
    p.precision = precision
    p.slab_order = slab_order
    p.tau = tau
    p.trt_lambda = trt_lambda
    return p


def _desc_array(descs):
    arr = (IoletDesc * max(len(descs), 1))()
    for i, d in enumerate(descs):
        arr[i] = d
    return arr


class Lattice:
    """One handle: LatticeData + LBM + BoundaryValues of the reference, on one GPU."""

    def __init__(self, geom: Geometry, prm: Params | None, inlets=(), outlets=()):
        """prm None: tables only; configure with set_params / set_iolets."""
        self._geom = geom
        self._inlets = list(inlets)
        self._outlets = list(outlets)
        v = geom.view()
        h = C.c_void_p()
        _check(lib().hlb_create(C.byref(v), C.byref(prm) if prm is not None else None,
                                _desc_array(self._inlets), len(self._inlets),
                                _desc_array(self._outlets), len(self._outlets), C.byref(h)))
        self._h = h
        self.n = int(lib().hlb_site_count(h))

    def set_params(self, prm: Params):
        _check(lib().hlb_set_params(self._h, C.byref(prm)))

    def get_params(self) -> Params:
        p = Params()
        _check(lib().hlb_get_params(self._h, C.byref(p)))
        return p

    def set_iolets(self, inlets=(), outlets=()):
        self._inlets = list(inlets)
        self._outlets = list(outlets)
        _check(lib().hlb_set_iolets(self._h, _desc_array(self._inlets), len(self._inlets),
                                    _desc_array(self._outlets), len(self._outlets)))

    def close(self):
        if getattr(self, "_h", None):
            lib().hlb_destroy(self._h)
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

    # -- tables ------------------------------------------------------------
    def class_counts(self) -> np.ndarray:
        out = np.zeros(6, dtype=np.int64)
        _check(lib().hlb_class_counts(self._h, _ptr(out)))
        return out

    def site_coords(self) -> np.ndarray:
        out = np.zeros((self.n, 3), dtype=np.int64)
        _check(lib().hlb_site_coords(self._h, _ptr(out)))
        return out

    def neighbour_tables(self):
        push = np.zeros((self.n, Q), dtype=np.int64)
        pull = np.zeros((18, self.n), dtype=np.uint32)
        _check(lib().hlb_neighbour_tables(self._h, _ptr(push), _ptr(pull)))
        return push, pull

    def site_masks(self):
        w = np.zeros(self.n, dtype=np.uint32)
        i = np.zeros(self.n, dtype=np.uint32)
        ident = np.zeros(self.n, dtype=np.int32)
        t = np.zeros(self.n, dtype=np.int32)
        _check(lib().hlb_site_masks(self._h, _ptr(w), _ptr(i), _ptr(ident), _ptr(t)))
        return w, i, ident, t

    def wall_geometry(self):
        d = np.zeros((self.n, 18), dtype=np.float64)
        nrm = np.zeros((self.n, 3), dtype=np.float64)
        _check(lib().hlb_wall_geometry(self._h, _ptr(d), _ptr(nrm)))
        return d, nrm

    # -- state ----------------------------------------------------------------
    def init_equilibrium(self, rho0=1.0, t0=1):
        _check(lib().hlb_init_equilibrium(self._h, rho0, t0))

    def upload_f(self, f: np.ndarray, t0=1):
        f = np.ascontiguousarray(f, dtype=np.float64).reshape(self.n, Q)
        _check(lib().hlb_upload_f(self._h, _ptr(f), t0))

    def step(self, nsteps: int, properties=False):
        _check(lib().hlb_step(self._h, nsteps, STEP_PROPERTIES if properties else 0))

    def step_timed(self, nsteps: int, properties=False) -> float:
        ms = C.c_double()
        _check(lib().hlb_step_timed(self._h, nsteps, STEP_PROPERTIES if properties else 0, C.byref(ms)))
        return ms.value

    def synchronize(self):
        _check(lib().hlb_synchronize(self._h))

    def download_f(self) -> np.ndarray:
        f = np.zeros((self.n, Q), dtype=np.float64)
        _check(lib().hlb_download_f(self._h, _ptr(f)))
        return f

    def fields(self):
        rho = np.zeros(self.n, dtype=np.float64)
        u = np.zeros((self.n, 3), dtype=np.float64)
        wss = np.zeros(self.n, dtype=np.float64)
        _check(lib().hlb_get_fields(self._h, _ptr(rho), _ptr(u), _ptr(wss)))
        return rho, u, wss

    def stress(self) -> np.ndarray:
        """Stress caches from the state entering the next step, n x 17: stress
        tensor (xx, xy, xz, yy, yz, zz), von Mises, shear rate, traction,
        tangential and normal projections of the traction."""
        rows = np.empty((self.n, 17))
        _check(lib().hlb_get_stress_rows(self._h, _ptr(rows)))
        return rows

    def timestep(self) -> int:
        return int(lib().hlb_timestep(self._h))

    def stable(self) -> bool:
        s = C.c_int()
        _check(lib().hlb_stability(self._h, C.byref(s)))
        return bool(s.value)

    def set_variant(self, variant: int):
        _check(lib().hlb_set_variant(self._h, variant))

    def set_sponge(self, viscosity_ratio: float, width: float, lifetime: int):
        """The LES kernel's sponge layer at the outlets (width in lattice units)."""
        _check(lib().hlb_set_sponge(self._h, float(viscosity_ratio), float(width), int(lifetime)))

    def set_graphs(self, enable: bool):
        """Replay captured step sequences (True, the default) or launch eagerly."""
        _check(lib().hlb_set_graphs(self._h, 1 if enable else 0))

    def captured_graphs(self) -> int:
        """Captured step sequences held for replay."""
        return int(lib().hlb_captured_graphs(self._h))

    def variant(self) -> int:
        return int(lib().hlb_variant(self._h))

    def autotune(self, trial_steps=20):
        v, ms = C.c_int(), C.c_double()
        _check(lib().hlb_autotune(self._h, trial_steps, C.byref(v), C.byref(ms)))
        return v.value, ms.value

    def monitor(self) -> dict:
        """Device reductions of the last property step: min/max density, max |u|, mass."""
        out = np.zeros(4, dtype=np.float64)
        _check(lib().hlb_monitor(self._h, _ptr(out)))
        return {"rho_min": out[0], "rho_max": out[1], "u_max": out[2], "mass": out[3]}

    def monitor_noalloc(self) -> dict:
        """monitor() computed in the library's fixed device scratch (no
        device allocation; calls that overlap on one GPU race)."""
        out = np.zeros(4, dtype=np.float64)
        _check(lib().hlb_monitor_noalloc(self._h, _ptr(out)))
        return {"rho_min": out[0], "rho_max": out[1], "u_max": out[2], "mass": out[3]}

    def iolet_state(self, outlet: bool, index: int) -> np.ndarray:
        """(density, densityNew, flowRate, flowRateOld) of one iolet."""
        out = np.zeros(4, dtype=np.float64)
        _check(lib().hlb_iolet_state(self._h, int(bool(outlet)), int(index), _ptr(out)))
        return out


    def checkpoint_read(self, path, target: int | None = None):
        """(timestep, f) of a distributions checkpoint record; the last one when
        target is None.  Restart with upload_f(f, timestep)."""
        n = int(lib().hlb_site_count(self._h))
        f = np.empty((n, Q), np.float64)
        t = C.c_int64()
        _check(lib().hlb_checkpoint_read(self._h, str(path).encode(), -1 if target is None else int(target),
                                         C.byref(t), _ptr(f)))
        return int(t.value), f


class Extraction:
    """A property-output file (.xtr, plus .off with distributions) of one lattice."""

    def __init__(self, lat: "Lattice", path, fields, selector=SELECT_WHOLE, voxel_size=1.0, time_step=1.0,
                 origin=(0.0, 0.0, 0.0), point=(0.0, 0.0, 0.0), normal=(0.0, 0.0, 1.0), radius=0.0, names=None,
                 point2=(0.0, 0.0, 0.0)):
        self._lat = lat
        self._fields = (C.c_int32 * len(fields))(*fields)
        self._names = None
        if names is not None:
            self._names = (C.c_char_p * len(fields))(*[None if n is None else n.encode() for n in names])
        spec = XtrSpec(C.cast(self._fields, C.POINTER(C.c_int32)),
                       None if self._names is None else C.cast(self._names, C.POINTER(C.c_char_p)),
                       len(fields), selector, voxel_size, time_step,
                       (C.c_double * 3)(*origin), (C.c_double * 3)(*point), (C.c_double * 3)(*normal), radius,
                       (C.c_double * 3)(*point2))
        h = C.c_void_p()
        _check(lib().hlb_xtr_open(lat._h, str(path).encode(), C.byref(spec), C.byref(h)))
        self._h = h

    def close(self):
        if getattr(self, "_h", None):
            lib().hlb_xtr_close(self._h)
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

    @property
    def site_count(self) -> int:
        return int(lib().hlb_xtr_site_count(self._h))

    def capture(self):
        _check(lib().hlb_xtr_capture(self._h))

    def write(self) -> int:
        t = C.c_int64()
        _check(lib().hlb_xtr_write(self._h, C.byref(t)))
        return int(t.value)

    def write_fields(self, timestep: int, rho=None, u=None, wss=None, f=None, stress=None):
        def p(a, shape):
            if a is None:
                return None
            a = np.ascontiguousarray(a, np.float64)
            assert a.size == int(np.prod(shape))
            return a
        n = int(lib().hlb_site_count(self._lat._h))
        arrs = [p(rho, (n,)), p(u, (n, 3)), p(wss, (n,)), p(f, (n, Q)), p(stress, (n, 17))]
        _check(lib().hlb_xtr_write_fields(self._h, int(timestep), *[None if a is None else _ptr(a) for a in arrs]))


class Batch:
    """Many FP32-shifted lattices advanced by one step launch per time step
    (hlb_batch_*).  Members stay owned by the caller."""

    def __init__(self, members=()):
        h = C.c_void_p()
        _check(lib().hlb_batch_create(C.byref(h)))
        self._h = h
        self._members = []
        for m in members:
            self.add(m)

    def close(self):
        if getattr(self, "_h", None):
            lib().hlb_batch_destroy(self._h)
            self._h = None
            self._members = []

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def add(self, lat: "Lattice"):
        _check(lib().hlb_batch_add(self._h, lat._h))
        self._members.append(lat)

    def remove(self, lat: "Lattice"):
        _check(lib().hlb_batch_remove(self._h, lat._h))
        self._members = [m for m in self._members if m is not lat]

    def size(self) -> int:
        return int(lib().hlb_batch_size(self._h))

    def sites(self) -> int:
        return int(lib().hlb_batch_sites(self._h))

    def step(self, nsteps: int, properties=False):
        _check(lib().hlb_batch_step(self._h, nsteps, STEP_PROPERTIES if properties else 0))

    def step_timed(self, nsteps: int, properties=False) -> float:
        ms = C.c_double()
        _check(lib().hlb_batch_step_timed(self._h, nsteps, STEP_PROPERTIES if properties else 0, C.byref(ms)))
        return ms.value

    def set_graphs(self, enable: bool):
        _check(lib().hlb_batch_set_graphs(self._h, 1 if enable else 0))

    def captured_graphs(self) -> int:
        """Captured step sequences held for replay."""
        return int(lib().hlb_batch_captured_graphs(self._h))

    def set_variant(self, variant: int):
        _check(lib().hlb_batch_set_variant(self._h, variant))

    def variant(self) -> int:
        return int(lib().hlb_batch_variant(self._h))

    def autotune(self, trial_steps=20):
        v = C.c_int()
        ms = C.c_double()
        _check(lib().hlb_batch_autotune(self._h, trial_steps, C.byref(v), C.byref(ms)))
        return v.value, ms.value


class Server:
    """The solve-request loop (hlb_server_*): continuous batching of
    FP32-shifted requests under a device-memory budget, or (plain=True) one
    request at a time in arrival order, each stepped alone.  submit() may be
    called from another thread than advance()."""

    def __init__(self, budget_bytes: int, quantum_steps: int = 100, plain: bool = False):
        h = C.c_void_p()
        _check(lib().hlb_server_create(int(budget_bytes), int(quantum_steps), C.byref(h)))
        self._h = h
        self.quantum = quantum_steps
        if plain:
            _check(lib().hlb_server_set_mode(h, SERVE_PLAIN))

    def close(self):
        if getattr(self, "_h", None):
            lib().hlb_server_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def submit(self, geom: Geometry, prm: Params, inlets=(), outlets=(), max_steps=1000, period=0,
               tolerance=0.0, rho0=1.0) -> int:
        view = geom.view()
        ins, outs = _desc_array(inlets), _desc_array(outlets)
        r = Request()
        r.geom = C.pointer(view)
        r.params = prm
        r.inlets = C.cast(ins, C.POINTER(IoletDesc)) if ins is not None else None
        r.n_inlets = len(inlets)
        r.outlets = C.cast(outs, C.POINTER(IoletDesc)) if outs is not None else None
        r.n_outlets = len(outlets)
        r.max_steps, r.period, r.tolerance, r.rho0 = int(max_steps), int(period), float(tolerance), float(rho0)
        rid = C.c_int64()
        _check(lib().hlb_server_submit(self._h, C.byref(r), C.byref(rid)))
        return rid.value

    def advance(self):
        run, q = C.c_int(), C.c_int()
        _check(lib().hlb_server_advance(self._h, C.byref(run), C.byref(q)))
        return run.value, q.value

    def status(self, rid: int) -> RequestStatus:
        st = RequestStatus()
        _check(lib().hlb_server_status(self._h, rid, C.byref(st)))
        return st

    def fields(self, rid: int):
        n = self.status(rid).sites
        rho, u, wss = np.zeros(n), np.zeros((n, 3)), np.zeros(n)
        _check(lib().hlb_server_fields(self._h, rid, _ptr(rho), _ptr(u), _ptr(wss)))
        return rho, u, wss

    def release(self, rid: int):
        _check(lib().hlb_server_release(self._h, rid))

    def site_steps(self) -> int:
        return int(lib().hlb_server_site_steps(self._h))

    def bytes_in_use(self) -> int:
        return int(lib().hlb_server_bytes_in_use(self._h))
