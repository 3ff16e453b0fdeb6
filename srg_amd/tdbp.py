"""ctypes binding of libsrg_tdbp.so (include/tdbp.h) and thin host helpers.

The library is the product: every compute call here goes to HIP kernels on
the GPU.  There is no CPU fallback -- if the library is missing, or no gfx950
device is visible, the calls raise.
"""
from __future__ import annotations

import ctypes as C
import math
import os
from dataclasses import dataclass, field
from typing import Optional

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("TDBP_LIB") or os.path.join(_HERE, "libsrg_tdbp.so")

# tdbp_status
OK, ERR_ARG, ERR_HIP, ERR_NODEV, ERR_IO, ERR_NOMEM, ERR_LIMIT = range(7)
# tdbp_precision
PLAIN_FP64, MIXED = 0, 1
# tdbp_dtype
CF32, CF16, CBF16, CI16 = 0, 1, 2, 3
# Arithmetic of the reference GPU entry (FP32 lerp, 1/N output scale, |Re| >
# 1e-18 merge) or of its CPU twin (FP64 lerp, unscaled, 1 <= |Re| < 2^31).
SEM_GPU, SEM_CPU = 0, 1
DTYPE_NAMES = {CF32: "cf32", CF16: "cf16", CBF16: "cbf16", CI16: "ci16"}


class TdbpError(RuntimeError):
    def __init__(self, code: int, msg: str):
        super().__init__(f"tdbp error {code}: {msg}")
        self.code = code


class Geom(C.Structure):
    """Mirror of tdbp_geom."""

    _fields_ = [
        ("rawdatalines", C.c_int32),
        ("samples", C.c_int32),
        ("aperture", C.c_int32),
        ("numstatevec", C.c_int32),
        ("rngstart", C.c_double),
        ("rngend", C.c_double),
        ("dmrg", C.c_double),
        ("wvl", C.c_double),
        ("prf", C.c_double),
        ("angc0", C.c_double),
        ("angc1", C.c_double),
        ("tmid", C.c_double),
        ("xyz_mid", C.c_double * 3),
        ("vel_mid", C.c_double * 3),
        ("timeorbit", C.POINTER(C.c_double)),
        ("xx", C.POINTER(C.c_double)),
        ("vv", C.POINTER(C.c_double)),
        ("demwidth", C.c_int32),
        ("firstline", C.c_int32),
        ("nlines", C.c_int32),
        ("firstpix", C.c_int32),
        ("lastpix", C.c_int32),
        ("firstlat", C.c_double),
        ("firstlon", C.c_double),
        ("deltalat", C.c_double),
        ("deltalon", C.c_double),
        ("fit_last_line", C.c_int32),
        ("semantics", C.c_int32),
    ]


class Chirp(C.Structure):
    """Mirror of tdbp_chirp."""

    _fields_ = [("rangedecimation", C.c_int32), ("nsamps", C.c_int32), ("npts", C.c_int32),
                ("nvalid", C.c_int32), ("samplefreq", C.c_float), ("ramprate", C.c_float),
                ("startfreq", C.c_float), ("pulselength", C.c_float)]

    def as_dict(self):
        return {k: getattr(self, k) for k, _ in self._fields_}


class BurstParams(C.Structure):
    """Mirror of tdbp_burst_params."""

    _fields_ = [("starttime", C.c_double), ("prf", C.c_double), ("samplefreq", C.c_double),
                ("pri", C.c_double), ("swst", C.c_double), ("range0", C.c_double),
                ("wvl", C.c_double), ("rangedecimation", C.c_int32), ("rank", C.c_int32)]

    def as_dict(self):
        return {k: getattr(self, k) for k, _ in self._fields_}


class Samples(C.Structure):
    """Mirror of tdbp_samples."""

    _fields_ = [("d_data", C.c_void_p), ("d_scale", C.c_void_p), ("dtype", C.c_int32)]


_lib = None

_VP = C.c_void_p
_DP = C.POINTER(C.c_double)
_IP = C.POINTER(C.c_int)
_GP = C.POINTER(Geom)
# The 33 by-reference arguments of azimuth_compress_ / azimuth_compress_cpu_
# (sentinel/azimuth_compress.cu:181-214).
_DROPIN_ARGS = [_VP, _DP, _IP, _IP, _IP, _IP, _IP, _IP, _DP, _DP, _DP, _DP, _DP, _DP, _DP,
                _DP, _IP, _DP, _DP, _DP, _DP, _DP, _DP, _DP, _DP, _DP, _DP, _DP, _IP, _IP,
                _DP, _DP, _DP]
_SP = C.POINTER(Samples)


def _sig(lib):
    sigs = {
        "tdbp_last_error": (C.c_char_p, []),
        "tdbp_device_count": (C.c_int, []),
        "tdbp_init": (C.c_int, [C.c_int]),
        "tdbp_dropin_status": (C.c_int, []),
        "tdbp_dropin_flush": (C.c_int, []),
        "tdbp_dev_alloc": (_VP, [C.c_size_t]),
        "tdbp_dev_free": (C.c_int, [_VP]),
        "tdbp_memcpy_htod": (C.c_int, [_VP, _VP, C.c_size_t, _VP]),
        "tdbp_memcpy_htod_staged": (C.c_int, [_VP, _VP, C.c_size_t, _VP]),
        "tdbp_memcpy_dtoh": (C.c_int, [_VP, _VP, C.c_size_t, _VP]),
        "tdbp_memcpy_dtod": (C.c_int, [_VP, _VP, C.c_size_t, _VP]),
        "tdbp_dev_zero": (C.c_int, [_VP, C.c_size_t, _VP]),
        "tdbp_dev_copy": (C.c_int, [_VP, _VP, C.c_size_t, _VP]),
        "tdbp_stream_create": (C.c_int, [C.POINTER(_VP)]),
        "tdbp_stream_destroy": (C.c_int, [_VP]),
        "tdbp_stream_sync": (C.c_int, [_VP]),
        "tdbp_stream_wait_event": (C.c_int, [_VP, _VP]),
        "tdbp_device_sync": (C.c_int, []),
        "tdbp_event_create": (C.c_int, [C.POINTER(_VP)]),
        "tdbp_event_destroy": (C.c_int, [_VP]),
        "tdbp_event_record": (C.c_int, [_VP, _VP]),
        "tdbp_event_elapsed_ms": (C.c_int, [_VP, _VP, C.POINTER(C.c_float)]),
        "tdbp_mem_info": (C.c_int, [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]),
        "tdbp_window": (None, [_DP, C.c_double, C.c_double, C.c_double, C.c_double,
                               C.c_int, C.c_int, _IP, _IP, _IP, _IP]),
        "tdbp_orbit_interp": (C.c_int, [_DP, _DP, _DP, C.c_int, _DP, C.c_int, _DP, _DP]),
        "tdbp_setxyz": (C.c_int, [_GP, _VP, _VP, _VP, _VP]),
        "tdbp_fit_aperture": (C.c_int, [_GP, _VP, _VP, _VP]),
        "tdbp_setazoff": (C.c_int, [_GP, _VP, _VP, _VP]),
        "tdbp_pair_count": (C.c_int, [_GP, _VP, _VP, _VP]),
        "tdbp_pack_samples": (C.c_int, [_VP, C.c_int, C.c_int, C.c_int, _VP, _VP, _VP]),
        "tdbp_chirp_decode": (C.c_int, [_VP, C.POINTER(Chirp)]),
        "tdbp_burst_decode": (C.c_int, [_VP, C.POINTER(BurstParams)]),
        "tdbp_steering_fit": (C.c_int, [_VP, C.c_size_t, C.c_int, _DP, _DP]),
        "tdbp_aperture": (C.c_int, [_DP, C.c_double, C.c_double, C.c_double, C.c_double]),
        "tdbp_bounds": (C.c_int, [C.c_double, C.c_double, C.c_double, C.c_double, _DP, _DP,
                                  _DP, C.c_int, _DP]),
        "tdbp_headers_dtoh": (C.c_int, [_VP, C.c_int, C.c_int, _VP, _VP]),
        "tdbp_burst_setup": (C.c_int, [_VP, C.c_size_t, C.c_int, C.c_int, _DP, _DP, _DP, _DP,
                                       C.c_int, C.c_int, C.c_int, C.c_double, C.c_double,
                                       C.c_double, C.c_double, _GP, _DP, _IP]),
        "tdbp_pulse_orbit": (C.c_int, [_VP, C.c_int, C.c_int, _DP, _DP, _DP, C.c_int, C.c_int,
                                       _VP, _VP, _VP, _VP]),
        "tdbp_crossmul": (C.c_int, [_VP, _VP, C.c_int, C.c_int, C.c_float, C.c_int, C.c_int,
                                    C.c_int, _VP, _VP, _VP]),
        "tdbp_makecc": (C.c_int, [_VP, _VP, C.c_int, C.c_int, _VP, _VP]),
        "tdbp_synth_raw": (C.c_int, [_VP, C.c_int, C.c_int, C.POINTER(Chirp), _VP, _DP, _DP,
                                     _VP, C.c_int, C.c_float, C.c_uint64, _VP]),
        "tdbp_range_compress": (C.c_int, [_VP, C.c_int, C.c_int, C.POINTER(Chirp), _VP,
                                          C.c_int, C.c_int, _VP, _VP, C.c_int, _VP]),
        "tdbp_headers_htod": (C.c_int, [_VP, C.c_int, C.c_int, _VP, _VP]),
        "tdbp_pixelint": (C.c_int, [_GP, _VP, _VP, _VP, _VP, _VP, _VP]),
        "tdbp_backproject": (C.c_int, [_GP, _SP, _VP, _VP, _VP, _VP, C.c_int, _VP]),
        "tdbp_backproject_variant": (C.c_int, [_GP, _SP, _VP, _VP, _VP, _VP, C.c_int,
                                               C.c_int, _VP]),
        "tdbp_backproject_noalloc": (C.c_int, [_GP, _SP, _VP, _VP, _VP, C.c_int, _VP]),
        "tdbp_autotune": (C.c_int, [_GP, _SP, _VP, _VP, _VP, C.c_int, C.c_int,
                                    C.POINTER(C.c_float), _IP]),
        "tdbp_set_variant": (C.c_int, [C.c_int]),
        "tdbp_variant_count": (C.c_int, []),
        "tdbp_variant_info": (C.c_int, [C.c_int, _IP, _IP, _IP]),
        "tdbp_batch_create": (_VP, [C.c_int, C.c_int]),
        "tdbp_batch_add": (C.c_int, [_VP, _GP, _SP, _VP, _VP, _VP]),
        "tdbp_batch_run": (C.c_int, [_VP, _VP]),
        "tdbp_batch_set_merge": (C.c_int, [_VP, C.c_int, _VP, C.c_int, C.c_int, C.c_int]),
        "tdbp_dropin_timing": (C.c_int, [C.POINTER(C.c_double), C.c_int]),
        "tdbp_compare": (C.c_int, [_VP, _VP, C.c_size_t, C.POINTER(C.c_double), _VP]),
        "tdbp_merge_geo": (C.c_int, [_VP, C.c_int, C.c_int, C.c_int, C.c_int, _VP, C.c_int,
                                     _VP]),
        "tdbp_batch_pairs": (C.c_int64, [_VP]),
        "tdbp_batch_variant": (C.c_int, [_VP]),
        "tdbp_batch_autotune": (C.c_int, [_VP, C.c_int, C.POINTER(C.c_float),
                                          C.POINTER(C.c_int)]),
        "tdbp_batch_device_bytes": (C.c_size_t, [_VP]),
        "tdbp_batch_destroy": (None, [_VP]),
        "tdbp_synth_clutter": (C.c_int, [_VP, C.c_int, C.c_int, C.c_uint64, C.c_float,
                                         C.POINTER(C.c_float), C.c_int, _VP]),
        "tdbp_synth_targets": (C.c_int, [_VP, _GP, _VP, _DP, C.POINTER(C.c_float),
                                         C.c_int, C.c_float, C.c_int, _VP]),
        "azimuth_compress_": (None, _DROPIN_ARGS),
        "azimuth_compress_cpu_": (None, _DROPIN_ARGS),
    }
    for name, (res, args) in sigs.items():
        f = getattr(lib, name)
        f.restype = res
        f.argtypes = args
    return lib


def exported_symbols():
    """Names of the entry points the binding declares (all must exist)."""
    return [
        "tdbp_last_error", "tdbp_device_count", "tdbp_init", "tdbp_dropin_status", "tdbp_dropin_flush",
        "tdbp_dev_alloc", "tdbp_dev_free", "tdbp_memcpy_htod", "tdbp_memcpy_htod_staged",
        "tdbp_memcpy_dtoh",
        "tdbp_memcpy_dtod", "tdbp_dev_zero", "tdbp_dev_copy", "tdbp_stream_create", "tdbp_stream_destroy",
        "tdbp_stream_sync", "tdbp_stream_wait_event", "tdbp_device_sync", "tdbp_event_create", "tdbp_event_destroy",
        "tdbp_event_record", "tdbp_event_elapsed_ms", "tdbp_mem_info", "tdbp_window",
        "tdbp_orbit_interp", "tdbp_setxyz", "tdbp_fit_aperture", "tdbp_setazoff",
        "tdbp_pair_count", "tdbp_pack_samples", "tdbp_chirp_decode", "tdbp_range_compress", "tdbp_synth_raw", "tdbp_crossmul",
        "tdbp_makecc", "tdbp_burst_decode", "tdbp_steering_fit", "tdbp_aperture", "tdbp_bounds",
        "tdbp_pulse_orbit", "tdbp_headers_dtoh", "tdbp_burst_setup", "tdbp_headers_htod", "tdbp_pixelint", "tdbp_backproject",
        "tdbp_backproject_variant", "tdbp_backproject_noalloc", "tdbp_autotune",
        "tdbp_set_variant",
        "tdbp_variant_count", "tdbp_variant_info", "tdbp_batch_create", "tdbp_batch_add",
        "tdbp_batch_run", "tdbp_batch_set_merge", "tdbp_merge_geo", "tdbp_compare", "tdbp_dropin_timing", "tdbp_batch_pairs",
        "tdbp_batch_variant", "tdbp_batch_autotune",
        "tdbp_batch_device_bytes", "tdbp_batch_destroy", "tdbp_synth_clutter",
        "tdbp_synth_targets", "azimuth_compress_", "azimuth_compress_cpu_",
    ]


def lib():
    """Load the HIP library (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise TdbpError(ERR_NODEV, f"{LIB_PATH} not built (run __graft_entry__.build())")
        _lib = _sig(C.CDLL(LIB_PATH))
    return _lib


def check(code: int):
    if code != OK:
        raise TdbpError(code, lib().tdbp_last_error().decode(errors="replace"))


def init(device: int = 0):
    check(lib().tdbp_init(device))


def _dp(a: np.ndarray):
    return a.ctypes.data_as(_DP)


# ----------------------------------------------------------------- memory


class DeviceArray:
    """A device allocation with a shape and dtype (numpy-like metadata)."""

    def __init__(self, shape, dtype):
        self.shape = tuple(int(s) for s in np.atleast_1d(shape))
        self.dtype = np.dtype(dtype)
        self.nbytes = int(np.prod(self.shape, dtype=np.int64)) * self.dtype.itemsize
        p = lib().tdbp_dev_alloc(self.nbytes)
        if not p:
            check(ERR_NOMEM)
        self.ptr = p
        self._base = None

    def rows(self, first: int, count: int) -> "DeviceArray":
        """View of rows [first, first + count) along the first axis; it shares
        this allocation and frees nothing."""
        if first < 0 or count < 1 or first + count > self.shape[0]:
            raise ValueError(f"rows [{first}, {first + count}) of {self.shape}")
        v = object.__new__(DeviceArray)
        v.shape = (count,) + self.shape[1:]
        v.dtype = self.dtype
        row = self.nbytes // self.shape[0]
        v.nbytes = row * count
        v.ptr = self.ptr + row * first
        v._base = self
        return v

    @classmethod
    def from_host(cls, a: np.ndarray, stream=None):
        a = np.ascontiguousarray(a)
        d = cls(a.shape, a.dtype)
        check(lib().tdbp_memcpy_htod(d.ptr, a.ctypes.data, a.nbytes, _s(stream)))
        return d

    def upload(self, a: np.ndarray, stream=None):
        a = np.ascontiguousarray(a, dtype=self.dtype)
        assert a.nbytes == self.nbytes
        check(lib().tdbp_memcpy_htod(self.ptr, a.ctypes.data, a.nbytes, _s(stream)))

    def upload_staged(self, a: np.ndarray, stream=None):
        """Upload from pageable memory through the library's pinned staging
        chunks; returns when `a` may be reused (the last DMAs may still run on
        `stream`)."""
        a = np.ascontiguousarray(a, dtype=self.dtype)
        assert a.nbytes == self.nbytes
        check(lib().tdbp_memcpy_htod_staged(self.ptr, a.ctypes.data, a.nbytes, _s(stream)))

    def download(self, stream=None) -> np.ndarray:
        out = np.empty(self.shape, self.dtype)
        check(lib().tdbp_memcpy_dtoh(out.ctypes.data, self.ptr, self.nbytes, _s(stream)))
        return out

    def zero(self, stream=None):
        check(lib().tdbp_dev_zero(self.ptr, self.nbytes, _s(stream)))

    def free(self):
        if self.ptr and self._base is None:
            lib().tdbp_dev_free(self.ptr)
        self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class Stream:
    def __init__(self):
        s = C.c_void_p()
        check(lib().tdbp_stream_create(C.byref(s)))
        self.ptr = s.value

    def sync(self):
        check(lib().tdbp_stream_sync(self.ptr))

    def wait(self, event: "Event"):
        """Later work on this stream waits for `event`."""
        check(lib().tdbp_stream_wait_event(self.ptr, event.ptr))

    def __del__(self):
        try:
            if self.ptr:
                lib().tdbp_stream_destroy(self.ptr)
        except Exception:
            pass


class Event:
    def __init__(self):
        e = C.c_void_p()
        check(lib().tdbp_event_create(C.byref(e)))
        self.ptr = e.value

    def record(self, stream=None):
        check(lib().tdbp_event_record(self.ptr, getattr(stream, "ptr", stream)))

    def elapsed_ms(self, later: "Event") -> float:
        ms = C.c_float()
        check(lib().tdbp_event_elapsed_ms(self.ptr, later.ptr, C.byref(ms)))
        return ms.value

    def __del__(self):
        try:
            if self.ptr:
                lib().tdbp_event_destroy(self.ptr)
        except Exception:
            pass


def sync():
    check(lib().tdbp_device_sync())


def mem_info():
    f, t = C.c_size_t(), C.c_size_t()
    check(lib().tdbp_mem_info(C.byref(f), C.byref(t)))
    return f.value, t.value


# ----------------------------------------------------------------- geometry


@dataclass
class BurstGeometry:
    """Host description of one burst and its DEM window (see tdbp_geom)."""

    L: int
    S: int
    A: int
    rngstart: float
    rngend: float
    dmrg: float
    wvl: float
    prf: float
    angc0: float
    angc1: float
    tmid: float
    xyz_mid: np.ndarray
    vel_mid: np.ndarray
    timeorbit: np.ndarray
    xx: np.ndarray
    vv: np.ndarray
    demwidth: int
    firstline: int
    nlines: int
    firstpix: int
    lastpix: int
    firstlat: float
    firstlon: float
    deltalat: float
    deltalon: float
    fit_last_line: int = 0
    semantics: int = 0
    _keep: list = field(default_factory=list, repr=False)

    def to_c(self) -> Geom:
        t = np.ascontiguousarray(self.timeorbit, np.float64)
        x = np.ascontiguousarray(self.xx, np.float64)
        v = np.ascontiguousarray(self.vv, np.float64)
        self._keep = [t, x, v]
        g = Geom()
        g.rawdatalines, g.samples, g.aperture = self.L, self.S, self.A
        g.numstatevec = len(t)
        g.rngstart, g.rngend, g.dmrg, g.wvl = self.rngstart, self.rngend, self.dmrg, self.wvl
        g.prf, g.angc0, g.angc1, g.tmid = self.prf, self.angc0, self.angc1, self.tmid
        for i in range(3):
            g.xyz_mid[i] = float(self.xyz_mid[i])
            g.vel_mid[i] = float(self.vel_mid[i])
        g.timeorbit, g.xx, g.vv = _dp(t), _dp(x), _dp(v)
        g.demwidth, g.firstline, g.nlines = self.demwidth, self.firstline, self.nlines
        g.firstpix, g.lastpix = self.firstpix, self.lastpix
        g.firstlat, g.firstlon = self.firstlat, self.firstlon
        g.deltalat, g.deltalon = self.deltalat, self.deltalon
        g.fit_last_line = self.fit_last_line
        g.semantics = self.semantics
        return g

    @property
    def nfit(self) -> int:
        return self.nlines if self.fit_last_line else self.nlines - 1


def window(latlons, firstlat, firstlon, deltalat, deltalon, demwidth, demlength):
    ll = np.ascontiguousarray(latlons, np.float64)
    out = [C.c_int() for _ in range(4)]
    lib().tdbp_window(_dp(ll), firstlat, firstlon, deltalat, deltalon, demwidth,
                      demlength, *[C.byref(o) for o in out])
    return tuple(o.value for o in out)


def orbit_interp(timeorbit, xx, vv, times):
    """Hermite positions and velocities at `times` (host code of the library)."""
    t = np.ascontiguousarray(timeorbit, np.float64)
    x = np.ascontiguousarray(xx, np.float64)
    v = np.ascontiguousarray(vv, np.float64)
    tm = np.ascontiguousarray(np.atleast_1d(times), np.float64)
    pos = np.empty((len(tm), 3))
    vel = np.empty((len(tm), 3))
    check(lib().tdbp_orbit_interp(_dp(t), _dp(x), _dp(v), len(t), _dp(tm), len(tm),
                                  _dp(pos), _dp(vel)))
    return pos, vel


# ------------------------------------------------------------ operators


def _s(stream):
    return getattr(stream, "ptr", stream)


def samples(d_data: DeviceArray, dtype=CF32, d_scale: Optional[DeviceArray] = None):
    s = Samples()
    s.d_data = d_data.ptr
    s.d_scale = d_scale.ptr if d_scale is not None else None
    s.dtype = dtype
    return s


def fit_aperture(g: BurstGeometry, d_dem: DeviceArray, d_coef: DeviceArray, stream=None):
    gc = g.to_c()
    check(lib().tdbp_fit_aperture(C.byref(gc), d_dem.ptr, d_coef.ptr, _s(stream)))


def setxyz(g: BurstGeometry, d_dem, d_xyz, d_xyzfit=None, stream=None):
    gc = g.to_c()
    check(lib().tdbp_setxyz(C.byref(gc), d_dem.ptr, d_xyz.ptr,
                            d_xyzfit.ptr if d_xyzfit is not None else None, _s(stream)))


def setazoff(g: BurstGeometry, d_coef, d_azoff, stream=None):
    gc = g.to_c()
    check(lib().tdbp_setazoff(C.byref(gc), d_coef.ptr, d_azoff.ptr, _s(stream)))


def pair_count(g: BurstGeometry, d_coef, d_pairs, stream=None):
    gc = g.to_c()
    check(lib().tdbp_pair_count(C.byref(gc), d_coef.ptr, d_pairs.ptr, _s(stream)))


def pixelint(g: BurstGeometry, d_burst, d_satloc, d_xyz, d_azoff, d_out, stream=None):
    gc = g.to_c()
    check(lib().tdbp_pixelint(C.byref(gc), d_burst.ptr, d_satloc.ptr, d_xyz.ptr,
                              d_azoff.ptr, d_out.ptr, _s(stream)))


def pack(d_cf32: DeviceArray, L: int, S: int, dtype: int, stream=None):
    """cf32 samples [L][S] -> (CF16/CBF16/CI16 words [L][S], FP32 scales [L])
    (tdbp_pack_samples): power-of-two scales, one common scale for the pulses
    within 2^16 (CF16/CBF16) or 2^4 (CI16) of the largest, value = word x
    scale."""
    if d_cf32.nbytes < L * S * 8:
        raise ValueError("pack: input smaller than L x S cf32 samples")
    d_packed = DeviceArray((L, S), np.uint32)
    d_scale = DeviceArray((L,), np.float32)
    check(lib().tdbp_pack_samples(d_cf32.ptr, L, S, dtype, d_packed.ptr, d_scale.ptr,
                                  _s(stream)))
    return d_packed, d_scale


def pack_into(d_cf32: DeviceArray, L: int, S: int, dtype: int, d_packed: DeviceArray,
              d_scale: DeviceArray, stream=None):
    """pack() into existing buffers (d_packed >= L*S words, d_scale >= L)."""
    if d_packed.nbytes < L * S * 4 or d_scale.nbytes < L * 4 or d_cf32.nbytes < L * S * 8:
        raise ValueError("pack_into: buffers smaller than L x S")
    check(lib().tdbp_pack_samples(d_cf32.ptr, L, S, dtype, d_packed.ptr, d_scale.ptr,
                                  _s(stream)))


def chirp_decode(header: bytes) -> Chirp:
    """Chirp parameters from an 80-byte packet header (host code, no device)."""
    h = np.frombuffer(bytes(header), np.uint8)
    if h.size < 80:
        raise ValueError("header needs 80 bytes")
    c = Chirp()
    check(lib().tdbp_chirp_decode(h.ctypes.data, C.byref(c)))
    return c


def burst_decode(header: bytes) -> BurstParams:
    """Burst parameters from a line's 80-byte header (host code)."""
    h = np.frombuffer(bytes(header), np.uint8)
    p = BurstParams()
    check(lib().tdbp_burst_decode(h.ctypes.data, C.byref(p)))
    return p


def steering_fit(headers: np.ndarray):
    """(angc0, angc1) from the headers of a burst's lines: uint8 [lines][>= 80]."""
    h = np.ascontiguousarray(headers, np.uint8)
    c0, c1 = C.c_double(), C.c_double()
    check(lib().tdbp_steering_fit(h.ctypes.data, h.shape[1], h.shape[0], C.byref(c0),
                                  C.byref(c1)))
    return c0.value, c1.value


def aperture(vel_mid_burst, range0: float, wvl: float, prf: float, angc1: float) -> int:
    v = np.ascontiguousarray(vel_mid_burst, np.float64)
    return int(lib().tdbp_aperture(v.ctypes.data_as(_DP), range0, wvl, prf, angc1))


def bounds(startime, endtime, startr, endr, timeorbit, xx, vv) -> np.ndarray:
    """[min lat, max lat, min lon, max lon] (deg) of a burst footprint."""
    t = np.ascontiguousarray(timeorbit, np.float64)
    x = np.ascontiguousarray(xx, np.float64).reshape(-1, 3)
    v = np.ascontiguousarray(vv, np.float64).reshape(-1, 3)
    out = np.zeros(4)
    dp = lambda a: a.ctypes.data_as(_DP)  # noqa: E731
    check(lib().tdbp_bounds(startime, endtime, startr, endr, dp(t), dp(x), dp(v), len(t),
                            dp(out)))
    return out


def headers_dtoh(d_lines: DeviceArray, stream=None) -> np.ndarray:
    """uint8 [nlines][80]: each decoded line's packet header."""
    nl, stride = d_lines.shape
    out = np.empty((nl, 80), np.uint8)
    check(lib().tdbp_headers_dtoh(d_lines.ptr, nl, stride, out.ctypes.data, _s(stream)))
    return out


def headers_htod(d_lines: DeviceArray, headers: np.ndarray, stream=None):
    """Write [nlines][80] header bytes into the device lines."""
    nl, stride = d_lines.shape
    h = np.ascontiguousarray(headers, np.uint8)
    if h.shape != (nl, 80):
        raise ValueError(f"headers {h.shape} for {nl} lines")
    check(lib().tdbp_headers_htod(d_lines.ptr, nl, stride, h.ctypes.data, _s(stream)))


def burst_setup(headers: np.ndarray, rangesamples: int, satvel_mid, timeorbit, xx, vv,
                demwidth: int, demlength: int, firstlat: float, firstlon: float,
                deltalat: float, deltalon: float):
    """(BurstGeometry, latlons, in_scene) of the driver's per-burst set-up."""
    h = np.ascontiguousarray(headers, np.uint8)
    t = np.ascontiguousarray(timeorbit, np.float64)
    x = np.ascontiguousarray(xx, np.float64).reshape(-1, 3)
    v = np.ascontiguousarray(vv, np.float64).reshape(-1, 3)
    sv = np.ascontiguousarray(satvel_mid, np.float64)
    g = Geom()
    ll = np.zeros(4)
    ins = C.c_int()
    dp = lambda a: a.ctypes.data_as(_DP)  # noqa: E731
    check(lib().tdbp_burst_setup(h.ctypes.data, h.shape[1], h.shape[0], rangesamples, dp(sv),
                                 dp(t), dp(x), dp(v), len(t), demwidth, demlength, firstlat,
                                 firstlon, deltalat, deltalon, C.byref(g), dp(ll),
                                 C.byref(ins)))
    geom = BurstGeometry(
        L=g.rawdatalines, S=g.samples, A=g.aperture, rngstart=g.rngstart, rngend=g.rngend,
        dmrg=g.dmrg, wvl=g.wvl, prf=g.prf, angc0=g.angc0, angc1=g.angc1, tmid=g.tmid,
        xyz_mid=np.array(g.xyz_mid[:]), vel_mid=np.array(g.vel_mid[:]), timeorbit=t, xx=x, vv=v,
        demwidth=g.demwidth, firstline=g.firstline, nlines=g.nlines, firstpix=g.firstpix,
        lastpix=g.lastpix, firstlat=g.firstlat, firstlon=g.firstlon, deltalat=g.deltalat,
        deltalon=g.deltalon, fit_last_line=g.fit_last_line)
    return geom, ll, bool(ins.value)


def pulse_orbit(d_lines: DeviceArray, timeorbit, xx, vv, quantize: bool = False, stream=None):
    """Per-line (satloc, satvel, times) device arrays from the header times."""
    nl, stride = d_lines.shape
    t = np.ascontiguousarray(timeorbit, np.float64)
    x = np.ascontiguousarray(xx, np.float64).reshape(-1, 3)
    v = np.ascontiguousarray(vv, np.float64).reshape(-1, 3)
    sat = DeviceArray((nl, 3), np.float64)
    vel = DeviceArray((nl, 3), np.float64)
    tim = DeviceArray((nl,), np.float64)
    dp = lambda a: a.ctypes.data_as(_DP)  # noqa: E731
    check(lib().tdbp_pulse_orbit(d_lines.ptr, nl, stride, dp(t), dp(x), dp(v), len(t),
                                 1 if quantize else 0, sat.ptr, vel.ptr, tim.ptr, _s(stream)))
    return sat, vel, tim


RC_ZERO_HEADER = 1


def range_compress(d_raw: DeviceArray, chirp: Chirp, d_out: Optional[DeviceArray] = None,
                   packed=None, stream=None, zero_header: bool = False):
    """Range compression of d_raw (cf32 [nlines][raw_stride], header in the
    first 10 samples).  d_out: cf32 [nlines][>= nvalid + 10] (header samples
    copied, or zero with zero_header); packed: (dtype, d_words [nlines]
    [nvalid + 10], d_scale [nlines])."""
    nlines, stride = d_raw.shape
    if d_out is not None and (d_out.shape[0] != nlines or d_out.dtype != np.complex64):
        raise ValueError("output must be cf32 with one row per line")
    dt, pw, ps = packed if packed is not None else (CF16, None, None)
    if pw is not None and (pw.nbytes < nlines * (chirp.nvalid + 10) * 4 or
                           ps.nbytes < nlines * 4):
        raise ValueError("packed output buffers too small")
    check(lib().tdbp_range_compress(
        d_raw.ptr, nlines, stride, C.byref(chirp), d_out.ptr if d_out is not None else None,
        d_out.shape[1] if d_out is not None else 0, RC_ZERO_HEADER if zero_header else 0,
        pw.ptr if pw is not None else None,
        ps.ptr if ps is not None else None, dt, _s(stream)))


def crossmul(d_img1: DeviceArray, d_img2: DeviceArray, nvalid: Optional[int] = None,
             scale: float = 1.0, looksac: int = 1, looksdn: int = 1, mask: bool = True,
             stream=None, out=None):
    """Interferogram and amplitude of two cf32 images [lines][na]
    (tdbp_crossmul); returns (d_igram, d_amp) [nvalid/looksdn][na/looksac],
    into `out` = (d_igram, d_amp) when given."""
    nl, na = d_img1.shape
    if d_img2.shape != d_img1.shape:
        raise ValueError("images differ in shape")
    nvalid = nl if nvalid is None else nvalid
    if nvalid > nl:
        raise ValueError(f"{nvalid} lines of a {nl}-line image")
    shape = (nvalid // looksdn, na // looksac)
    if out is not None:
        ig, am = out
        if ig.shape != shape or am.shape != shape:
            raise ValueError(f"outputs must be {shape}")
    else:
        ig = DeviceArray(shape, np.complex64)
        am = DeviceArray(shape, np.complex64)
    check(lib().tdbp_crossmul(d_img1.ptr, d_img2.ptr, na, nvalid, scale, looksac, looksdn,
                              1 if mask else 0, ig.ptr, am.ptr, _s(stream)))
    return ig, am


def makecc(d_igram: DeviceArray, d_amp: DeviceArray, stream=None) -> DeviceArray:
    """Amplitude and correlation rows [nlines][2 npix] (tdbp_makecc)."""
    nl, npix = d_igram.shape
    out = DeviceArray((nl, 2 * npix), np.float32)
    check(lib().tdbp_makecc(d_igram.ptr, d_amp.ptr, npix, nl, out.ptr, _s(stream)))
    return out


def backproject(g: BurstGeometry, smp: Samples, d_satloc, d_dem, d_out,
                precision=PLAIN_FP64, d_coef=None, variant=None, stream=None):
    gc = g.to_c()
    coef = d_coef.ptr if d_coef is not None else None
    if variant is None:
        check(lib().tdbp_backproject(C.byref(gc), C.byref(smp), d_satloc.ptr, d_dem.ptr,
                                     coef, d_out.ptr, precision, _s(stream)))
    else:
        check(lib().tdbp_backproject_variant(C.byref(gc), C.byref(smp), d_satloc.ptr,
                                             d_dem.ptr, coef, d_out.ptr, precision,
                                             variant, _s(stream)))


def backproject_noalloc(g: BurstGeometry, smp: Samples, d_satloc, d_dem, d_out,
                        precision=PLAIN_FP64, stream=None):
    """tdbp_backproject_noalloc: the burst with its own fit, no device
    allocation (scratch in the library's per-GPU array; <= 16384 lines)."""
    gc = g.to_c()
    check(lib().tdbp_backproject_noalloc(C.byref(gc), C.byref(smp), d_satloc.ptr, d_dem.ptr,
                                         d_out.ptr, precision, _s(stream)))


def autotune(g: BurstGeometry, smp: Samples, d_satloc, d_dem, d_out, precision=MIXED,
             reps=3):
    gc = g.to_c()
    n = lib().tdbp_variant_count()
    ms = (C.c_float * n)()
    best = C.c_int(-1)
    check(lib().tdbp_autotune(C.byref(gc), C.byref(smp), d_satloc.ptr, d_dem.ptr,
                              d_out.ptr, precision, reps, ms, C.byref(best)))
    return best.value, list(ms)


def variant_info(v: int):
    r, c, s = C.c_int(), C.c_int(), C.c_int()
    check(lib().tdbp_variant_info(v, C.byref(r), C.byref(c), C.byref(s)))
    return r.value, c.value, s.value


class Batch:
    """Many bursts in one persistent launch (tdbp_batch_*)."""

    def __init__(self, precision=MIXED, variant=-1):
        p = lib().tdbp_batch_create(precision, variant)
        if not p:
            check(ERR_ARG)
        self.ptr = p
        self._keep = []

    def add(self, g: BurstGeometry, smp: Samples, d_satloc, d_dem, d_out) -> int:
        gc = g.to_c()
        self._keep.append((g, smp, d_satloc, d_dem, d_out))
        r = lib().tdbp_batch_add(self.ptr, C.byref(gc), C.byref(smp), d_satloc.ptr,
                                 d_dem.ptr, d_out.ptr)
        if r < 0:
            check(-r)
        return r

    def set_merge(self, burst: int, d_grid: DeviceArray, firstline: int):
        check(lib().tdbp_batch_set_merge(self.ptr, burst, d_grid.ptr, d_grid.shape[0],
                                         d_grid.shape[1], firstline))

    def run(self, stream=None):
        check(lib().tdbp_batch_run(self.ptr, _s(stream)))

    def autotune(self, reps: int = 2):
        """Time every VALU variant on this batch (tdbp_batch_autotune) and keep
        the fastest for this batch (the process default is unchanged); returns
        (best, ms per variant), best -1 where the automatic choice over bursts
        of different sizes beats every variant."""
        n = lib().tdbp_variant_count()
        ms = (C.c_float * n)()
        best = C.c_int(-1)
        check(lib().tdbp_batch_autotune(self.ptr, reps, ms, C.byref(best)))
        return best.value, list(ms)

    @property
    def pairs(self) -> int:
        return int(lib().tdbp_batch_pairs(self.ptr))

    @property
    def variant(self) -> int:
        return int(lib().tdbp_batch_variant(self.ptr))

    @property
    def device_bytes(self) -> int:
        return int(lib().tdbp_batch_device_bytes(self.ptr))

    def close(self):
        if self.ptr:
            lib().tdbp_batch_destroy(self.ptr)
            self.ptr = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def merge_geo(d_grid: DeviceArray, firstline: int, d_out: DeviceArray, stream=None,
              semantics: int = SEM_GPU):
    """Merge a burst output [nlines][W] into grid rows [firstline, ...) with
    the .geo rule of the GPU entry or of the CPU twin."""
    nl, W = d_out.shape
    check(lib().tdbp_merge_geo(d_grid.ptr, W, d_grid.shape[0], firstline, nl, d_out.ptr,
                               semantics, _s(stream)))


def compare(d_img: DeviceArray, d_ref: DeviceArray, stream=None) -> dict:
    """RMS phase (rad) and relative amplitude error of a cf32 image against a
    cf32 reference over the reference's nonzero pixels, summed on the device;
    sum_w is the reference's power over those pixels (the weight that
    combines the errors of several images)."""
    if d_img.nbytes != d_ref.nbytes or d_img.dtype != np.complex64:
        raise ValueError("compare needs two cf32 arrays of one size")
    n = d_img.nbytes // 8
    sums = (C.c_double * 5)()
    check(lib().tdbp_compare(d_img.ptr, d_ref.ptr, n, sums, _s(stream)))
    w = sums[1]
    return {"phase_rms": math.sqrt(sums[0] / w) if w > 0 else 0.0,
            "amp_rms": math.sqrt(sums[2] / w) if w > 0 else 0.0,
            "pixels": int(sums[3]), "extra_nonzero": int(sums[4]), "sum_w": w}


def synth_raw(d_raw: DeviceArray, chirp: Chirp, header: bytes, delay, carrier, amp,
              noise: float, seed: int, stream=None):
    """Decoded echo lines of point targets (tdbp_synth_raw)."""
    L, stride = d_raw.shape
    dl = np.ascontiguousarray(delay, np.float64).reshape(L, -1)
    cr = np.ascontiguousarray(carrier, np.float64).reshape(L, -1)
    a = np.asarray(amp, np.complex128).ravel()
    af = np.ascontiguousarray(np.stack([a.real, a.imag], 1), np.float32)
    h = np.frombuffer(bytes(header), np.uint8)
    dp = lambda x: x.ctypes.data_as(_DP)  # noqa: E731
    check(lib().tdbp_synth_raw(d_raw.ptr, L, stride, C.byref(chirp), h.ctypes.data, dp(dl),
                               dp(cr), af.ctypes.data, len(a), noise, seed, _s(stream)))


def synth_clutter(d: DeviceArray, L: int, S: int, seed: int, sigma: float,
                  taps: np.ndarray, stream=None):
    t = np.ascontiguousarray(taps, np.float32)
    check(lib().tdbp_synth_clutter(d.ptr, L, S, seed, sigma,
                                   t.ctypes.data_as(C.POINTER(C.c_float)), len(t),
                                   _s(stream)))


def synth_targets(d: DeviceArray, g: BurstGeometry, d_satloc, xyz, amp, res=1.14,
                  halfwidth=16, stream=None):
    gc = g.to_c()
    x = np.ascontiguousarray(xyz, np.float64).reshape(-1, 3)
    a = np.empty((len(x), 2), np.float32)
    a[:, 0] = np.real(amp)
    a[:, 1] = np.imag(amp)
    check(lib().tdbp_synth_targets(d.ptr, C.byref(gc), d_satloc.ptr, _dp(x),
                                   a.ctypes.data_as(C.POINTER(C.c_float)), len(x),
                                   res, halfwidth, _s(stream)))
