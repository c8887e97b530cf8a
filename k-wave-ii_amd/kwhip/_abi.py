"""ctypes view of the C ABI in include/kwhip.h.

The product library is ``libkwhip.so`` (HIP, gfx950).  ``libkwhip_emu.so`` is
the same host code over the CPU lane emulator.  The public API always runs
the HIP library; the test-suite alone switches to the emulator, with the
private ``_backend_override`` context.  There is no silent fallback: if the
HIP library is missing, loading fails.
"""

from __future__ import annotations

import contextlib
import ctypes as C
import os
from pathlib import Path

import numpy as np

LIB_DIR = Path(__file__).resolve().parent / "_lib"
LIB_NAMES = {"hip": "libkwhip.so", "emu": "libkwhip_emu.so"}

KW_OK = 0
KW_EINVAL = -1
KW_EUNSUP = -2
KW_EDEVICE = -3
KW_ENOMEM = -4
KW_ESTATE = -5
KW_ENUMERIC = -6

REC = {
    "p": 1 << 0, "p_max": 1 << 1, "p_min": 1 << 2, "p_rms": 1 << 3,
    "p_max_all": 1 << 4, "p_min_all": 1 << 5, "p_final": 1 << 6,
    "u": 1 << 7, "u_max": 1 << 8, "u_min": 1 << 9, "u_rms": 1 << 10,
    "u_max_all": 1 << 11, "u_min_all": 1 << 12, "u_final": 1 << 13,
    "u_non_staggered": 1 << 14, "u_split_field": 1 << 15,
}
SRC_MODE = {"dirichlet": 0, "additive-no-correction": 1, "additive": 2}
NKINDS = 9
NOALLOC_MAX_BYTES = 128 << 20  # KW_NOALLOC_MAX_BYTES

c_double_p = C.POINTER(C.c_double)
c_float_p = C.POINTER(C.c_float)
c_u64_p = C.POINTER(C.c_uint64)


class TimeSource(C.Structure):
    _fields_ = [
        ("flag", C.c_int64),
        ("mode", C.c_int32),
        ("num_points", C.c_int64),
        ("index", c_u64_p),
        ("num_series", C.c_int64),
        ("sig_index", c_u64_p),
        ("input", c_double_p),
    ]


class Problem(C.Structure):
    _fields_ = [
        ("dim", C.c_int32),
        ("Nx", C.c_int64), ("Ny", C.c_int64), ("Nz", C.c_int64),
        ("Nt", C.c_int64),
        ("dx", C.c_double), ("dy", C.c_double), ("dz", C.c_double), ("dt", C.c_double),
        ("c_ref", C.c_double),
        ("c0", c_double_p), ("c0_scalar", C.c_double),
        ("rho0", c_double_p), ("rho0_scalar", C.c_double),
        ("rho0_sg", c_double_p * 3),
        ("nonlinear_flag", C.c_int32),
        ("BonA", c_double_p), ("BonA_scalar", C.c_double),
        ("absorbing_flag", C.c_int32),
        ("alpha_coeff", c_double_p), ("alpha_coeff_scalar", C.c_double),
        ("alpha_power", C.c_double),
        ("alpha_mode", C.c_int32),
        ("alpha_sign", C.c_double * 2),
        ("alpha_sign_set", C.c_int32),
        ("pml_size", C.c_int64 * 3),
        ("pml_alpha", C.c_double * 3),
        ("use_kspace", C.c_int32),
        ("use_sg", C.c_int32),
        ("p0", c_double_p),
        ("p_source", TimeSource),
        ("u_source", TimeSource * 3),
        ("sensor_num_points", C.c_int64),
        ("sensor_mask_index", c_u64_p),
        ("record_flags", C.c_uint32),
        ("record_start_index", C.c_int64),
        ("time_reversal_boundary_data", c_double_p),
        ("sensor_tri", c_u64_p), ("sensor_bc", c_double_p),
        ("directivity_angle", c_double_p), ("directivity_pattern", C.c_int32),
        ("directivity_size", C.c_double), ("alpha_filter", c_double_p),
        ("sensor_mask_corners", c_u64_p), ("sensor_num_cuboids", C.c_int64),
        ("axisymmetric", C.c_int32),
    ]


class Sizes(C.Structure):
    _fields_ = [("num_sensor_points", C.c_int64), ("num_recorded_time_points", C.c_int64),
                ("grid_cells", C.c_int64)]


# summed split density at the sensor points (the new toolbox's density sensor)
KW_REC_RHO = 1 << 16


class Outputs(C.Structure):
    _fields_ = [
        ("p", c_float_p), ("p_max", c_double_p), ("p_min", c_double_p), ("p_rms", c_double_p),
        ("p_max_all", c_double_p), ("p_min_all", c_double_p), ("p_final", c_float_p),
        ("u", c_float_p * 3), ("u_max", c_double_p * 3), ("u_min", c_double_p * 3),
        ("u_rms", c_double_p * 3), ("u_max_all", c_double_p * 3), ("u_min_all", c_double_p * 3),
        ("u_final", c_float_p * 3), ("u_non_staggered", c_float_p * 3),
        ("u_split_p", c_float_p * 3), ("u_split_s", c_float_p * 3), ("rho", c_float_p),
    ]


class KernelStats(C.Structure):
    _fields_ = [("ms", C.c_double * NKINDS), ("launches", C.c_int64 * NKINDS),
                ("bytes", C.c_double * NKINDS)]


class EngineConfig(C.Structure):
    _fields_ = [("device_bytes", C.c_int64), ("steps_per_round", C.c_int32),
                ("admit_threads", C.c_int32)]


class TicketInfo(C.Structure):
    _fields_ = [("status", C.c_int32), ("error", C.c_int32), ("submit_s", C.c_double),
                ("start_s", C.c_double), ("done_s", C.c_double), ("steps_done", C.c_int64),
                ("steps_total", C.c_int64), ("grid_cells", C.c_int64),
                ("device_bytes", C.c_int64)]


class EngineStats(C.Structure):
    _fields_ = [("submitted", C.c_int64), ("completed", C.c_int64), ("failed", C.c_int64),
                ("cancelled", C.c_int64), ("queued", C.c_int64), ("running", C.c_int64),
                ("device_bytes", C.c_int64), ("device_budget", C.c_int64),
                ("cell_steps", C.c_double), ("busy_s", C.c_double), ("launches", C.c_int64)]


TICKET_STATUS = {0: "queued", 1: "running", 2: "done", 3: "failed", 4: "cancelled"}


class KWError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__(f"kwhip error {code}: {msg}")
        self.code = code


_libs: dict[str, C.CDLL] = {}
_active = "hip"


def active_backend() -> str:
    """The library the public API runs: the HIP library, unless the
    test-suite has switched to the emulator build."""
    return _active


@contextlib.contextmanager
def _backend_override(name: str):
    """Test harness only: run the public API on another build of the library
    (``"emu"``: the CPU lane emulator) inside the ``with`` block."""
    global _active
    if name not in LIB_NAMES:
        raise ValueError(name)
    prev, _active = _active, name
    try:
        yield
    finally:
        _active = prev


def host_threads() -> int:
    """Host threads for the host-side precompute (FFT workers)."""
    return max(1, min(16, os.cpu_count() or 1))


def library_path(backend: str = "hip") -> Path:
    return LIB_DIR / LIB_NAMES[backend]


def load(backend: str = "hip") -> C.CDLL:
    """Load the kwhip library.  ``backend="hip"`` is the product; a missing
    library is an error (no fallback)."""
    if backend in _libs:
        return _libs[backend]
    path = library_path(backend)
    if not path.exists():
        raise ImportError(f"{path} is not built; run __graft_entry__.build() first")
    lib = C.CDLL(str(path))
    P = C.POINTER
    lib.kw_abi_version.restype = C.c_int
    lib.kw_backend.restype = C.c_char_p
    lib.kw_kind_name.restype = C.c_char_p
    lib.kw_kind_name.argtypes = [C.c_int]
    err = [C.c_char_p, C.c_size_t]
    lib.kw_output_sizes.argtypes = [P(Problem), P(Sizes)] + err
    lib.kw_run.argtypes = [P(Problem), P(Outputs)] + err
    lib.kw_run_noalloc.argtypes = [P(Problem), P(Outputs)] + err
    lib.kw_sim_create.argtypes = [P(Problem), P(C.c_void_p)] + err
    lib.kw_tiles.argtypes = [P(Problem), P(C.c_int32)] + err
    lib.kw_sim_extend.argtypes = [C.c_void_p, C.c_int64] + err
    lib.kw_sim_change_dt.argtypes = [C.c_void_p, C.c_double, C.c_double] + err
    lib.kw_sim_init_velocity.argtypes = [C.c_void_p, c_double_p * 3] + err
    lib.kw_sim_get_fields.argtypes = [C.c_void_p, c_float_p, c_float_p * 3, c_float_p * 3] + err
    lib.kw_sim_step.argtypes = [C.c_void_p, C.c_int64] + err
    lib.kw_sim_sync.argtypes = [C.c_void_p] + err
    lib.kw_sim_read.argtypes = [C.c_void_p, P(Outputs)] + err
    lib.kw_sim_steps_done.argtypes = [C.c_void_p]
    lib.kw_sim_steps_done.restype = C.c_int64
    lib.kw_sim_device_bytes.argtypes = [C.c_void_p]
    lib.kw_sim_device_bytes.restype = C.c_int64
    lib.kw_sim_destroy.argtypes = [C.c_void_p]
    lib.kw_sim_step_timed.argtypes = [C.c_void_p, C.c_int64, P(C.c_double), P(KernelStats)] + err
    lib.kw_smooth.argtypes = [C.c_int32, P(C.c_int64), c_double_p, c_double_p, c_double_p] + err
    lib.kw_layout_strided.argtypes = [C.c_int32, P(C.c_int64), P(C.c_int64), c_double_p,
                                      c_double_p, P(c_double_p)] + err
    lib.kw_save_problem.argtypes = [P(Problem), C.c_char_p] + err
    lib.kw_run_file.argtypes = [C.c_char_p, C.c_char_p, C.c_uint32, C.c_int64] + err
    lib.kw_engine_create.argtypes = [P(EngineConfig), P(C.c_void_p)] + err
    lib.kw_submit.argtypes = [C.c_void_p, P(Problem), P(C.c_int64)] + err
    lib.kw_poll.argtypes = [C.c_void_p, C.c_int64, P(TicketInfo)] + err
    lib.kw_wait.argtypes = [C.c_void_p, C.c_int64, P(Outputs)] + err
    lib.kw_cancel.argtypes = [C.c_void_p, C.c_int64] + err
    lib.kw_engine_get_stats.argtypes = [C.c_void_p, P(EngineStats)] + err
    lib.kw_engine_destroy.argtypes = [C.c_void_p]
    if lib.kw_abi_version() != 2:
        raise ImportError("kwhip ABI version mismatch")
    _libs[backend] = lib
    return lib


def call(fn, *args):
    buf = C.create_string_buffer(1024)
    rc = fn(*args, buf, C.c_size_t(len(buf)))
    if rc != KW_OK:
        raise KWError(rc, buf.value.decode(errors="replace"))


def dptr(a):
    """double* of a C-contiguous float64 array (None -> NULL)."""
    if a is None:
        return None
    return a.ctypes.data_as(c_double_p)


def fptr(a):
    if a is None:
        return None
    return a.ctypes.data_as(c_float_p)


def uptr(a):
    if a is None:
        return None
    return a.ctypes.data_as(c_u64_p)


def as_f64(a):
    return None if a is None else np.ascontiguousarray(a, dtype=np.float64)


def _layout(a, out, sg):
    if not a.flags.aligned or any(s % a.itemsize for s in a.strides):
        a = np.ascontiguousarray(a)
    sgp = None if sg is None else (c_double_p * 3)(*[dptr(s) for s in sg])
    sizes = (C.c_int64 * 3)(*a.shape, *([1] * (3 - a.ndim)))
    steps = (C.c_int64 * 3)(*[s // a.itemsize for s in a.strides], *([0] * (3 - a.ndim)))
    call(load(active_backend()).kw_layout_strided, C.c_int32(a.ndim), sizes, steps, dptr(a),
         dptr(out), sgp)


def fortran_flat(a):
    """Column-major (MATLAB) flattening of a grid array as float64; large
    grids in any other order (row-major, cut out of a larger array, axes
    exchanged or reversed) go through the library's threaded transpose."""
    a = np.asarray(a, dtype=np.float64)
    if a.ndim not in (2, 3) or a.size < (1 << 16) or a.flags.f_contiguous:
        return np.ascontiguousarray(a.ravel(order="F"))
    out = np.empty(a.size)
    _layout(a, out, None)
    return out


def fortran_staggered(a):
    """fortran_flat(a) and, per axis, the values half a cell further along it
    (v + 0.5 (v_next - v), the last plane unchanged), flattened alike."""
    a = np.asarray(a, dtype=np.float64)
    if a.size >= (1 << 16):
        sg = [np.empty(a.size) for _ in range(a.ndim)]
        # (a column-major grid is its own flattening)
        flat = fortran_flat(a) if a.flags.f_contiguous else np.empty(a.size)
        _layout(flat.reshape(a.shape, order="F") if a.flags.f_contiguous else a, flat, sg)
        return flat, sg
    sg = []
    for ax in range(a.ndim):
        s = a.copy()
        lo, hi = ((slice(None),) * ax + (slice(*r),) for r in ((0, -1), (1, None)))
        s[lo] = a[lo] + 0.5 * (a[hi] - a[lo])
        sg.append(fortran_flat(s))
    return fortran_flat(a), sg


def backend_name(lib) -> str:
    return lib.kw_backend().decode()


os.environ.setdefault("HSA_ENABLE_IPC_MODE_LEGACY", "0")
