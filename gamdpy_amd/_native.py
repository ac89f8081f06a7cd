"""ctypes binding of the C ABI declared in include/gamdpy_amd.h.

The shared library ``libgamdpy_amd.so`` is built in-tree by
``gamdpy_amd._build.build()``.  Nothing here falls back to a CPU
implementation: if the library is missing or the GPU is absent, the call
that needs it raises.
"""
import ctypes
import os
import threading

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libgamdpy_amd.so")
HEADER_PATH = os.path.join(os.path.dirname(_HERE), "include", "gamdpy_amd.h")

ABI_VERSION = 9

# enums of gamdpy_amd.h
PAIR_BASE = {"LJ_12_6_sigma_epsilon": 0, "LJ_12_6": 1, "IPL_n": 2, "LJ_m_n": 3, "harmonic_repulsion": 4,
             "hertzian": 5, "SAAP": 6, "sum": 7}
CUTOFF = {None: 0, "SP": 1, "SF": 2}
NBLIST = {"N squared": 0, "linked lists": 1}
INTEGRATOR = {None: 0, "NVE": 1, "NVT": 2, "NVT_Langevin": 3, "NPT_Atomic": 4}
TFUNC = {"constant": 0, "ramp": 1, "sin": 2}
SAVE_COLUMNS = ["U", "W", "lapU", "K", "Fsq", "Vol"]

c_float_p = ctypes.POINTER(ctypes.c_float)
c_int_p = ctypes.POINTER(ctypes.c_int)
c_u64_p = ctypes.POINTER(ctypes.c_ulonglong)


class GmdDesc(ctypes.Structure):
    """Mirror of ``gmd_desc`` (field order and types must match the header)."""
    _fields_ = [
        ("abi_version", ctypes.c_int),
        ("N", ctypes.c_int), ("D", ctypes.c_int), ("ntypes", ctypes.c_int),
        ("box", ctypes.c_float * 3),
        ("pair_base", ctypes.c_int), ("cutoff", ctypes.c_int),
        ("params", c_float_p),
        ("pair_exps", ctypes.c_float * 2),
        ("max_cut", ctypes.c_float),
        ("nparams", ctypes.c_int),
        ("nterms", ctypes.c_int),
        ("term_kind", ctypes.c_int * 2),
        ("term_first", ctypes.c_int * 2),
        ("term_exps", ctypes.c_float * 4),
        ("nblist_kind", ctypes.c_int),
        ("skin", ctypes.c_float),
        ("max_nbs", ctypes.c_int),
        ("utilize_niii", ctypes.c_int),
        ("exclusions", c_int_p),
        ("exclusions_cols", ctypes.c_int),
        ("integrator", ctypes.c_int),
        ("dt", ctypes.c_float),
        ("omega2", ctypes.c_float),
        ("degrees", ctypes.c_longlong),
        ("alpha", ctypes.c_float),
        ("seed", ctypes.c_ulonglong),
        ("tfunc", ctypes.c_int),
        ("tparams", ctypes.c_float * 4),
        ("compute_u", ctypes.c_int), ("compute_w", ctypes.c_int), ("compute_lap", ctypes.c_int),
        ("compute_k", ctypes.c_int), ("compute_fsq", ctypes.c_int),
        ("nscalars", ctypes.c_int), ("sid_u", ctypes.c_int), ("sid_w", ctypes.c_int), ("sid_lap", ctypes.c_int),
        ("sid_k", ctypes.c_int), ("sid_fsq", ctypes.c_int), ("sid_m", ctypes.c_int),
        ("momentum_reset_every", ctypes.c_int),
        ("scalar_save_every", ctypes.c_int),
        ("scalar_saves_per_block", ctypes.c_int),
        ("pb", ctypes.c_int), ("tp", ctypes.c_int), ("gridsync", ctypes.c_int),
        ("use_graph", ctypes.c_int),
        ("conf_saves_per_block", ctypes.c_int),
        ("nbonds", ctypes.c_int),
        ("bonds", c_int_p),
        ("nbond_types", ctypes.c_int),
        ("bond_params", c_float_p),
        ("mass_t", ctypes.c_float), ("mass_p", ctypes.c_float),
        ("pfunc", ctypes.c_int),
        ("pparams", ctypes.c_float * 4),
    ]


class GmdDeviceInfo(ctypes.Structure):
    _fields_ = [("compute_units", ctypes.c_int), ("wavefront_size", ctypes.c_int),
                ("max_threads_per_block", ctypes.c_int), ("total_mem", ctypes.c_longlong),
                ("name", ctypes.c_char * 64), ("arch", ctypes.c_char * 64)]


class GmdAdjDesc(ctypes.Structure):
    """Mirror of ``gmd_adj_desc`` (differentiable NVE trajectory)."""
    _fields_ = [("N", ctypes.c_int), ("ntypes", ctypes.c_int), ("box", ctypes.c_float * 3), ("dt", ctypes.c_float),
                ("nsteps", ctypes.c_int), ("ckpt_every", ctypes.c_int), ("rdf_every", ctypes.c_int),
                ("rdf_bins", ctypes.c_int), ("rdf_rmax", ctypes.c_float), ("rdf_width", ctypes.c_float)]


c_double_p = ctypes.POINTER(ctypes.c_double)

_SIGNATURES = {
    "gmd_abi_version": (ctypes.c_int, []),
    "gmd_desc_size": (ctypes.c_int, []),
    "gmd_last_error": (ctypes.c_char_p, []),
    "gmd_get_device_info": (ctypes.c_int, [ctypes.POINTER(GmdDeviceInfo)]),
    "gmd_create": (ctypes.c_int, [ctypes.POINTER(GmdDesc), ctypes.POINTER(ctypes.c_void_p)]),
    "gmd_destroy": (ctypes.c_int, [ctypes.c_void_p]),
    "gmd_upload": (ctypes.c_int, [ctypes.c_void_p, c_float_p, c_float_p, c_float_p, c_float_p, c_int_p, c_int_p]),
    "gmd_download": (ctypes.c_int, [ctypes.c_void_p, c_float_p, c_float_p, c_float_p, c_float_p, c_int_p, c_int_p]),
    "gmd_run": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_float, ctypes.c_int]),
    "gmd_evaluate": (ctypes.c_int, [ctypes.c_void_p]),
    "gmd_last_run_ms": (ctypes.c_int, [ctypes.c_void_p, c_float_p]),
    "gmd_profile_steps": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_float, ctypes.c_int, c_float_p, c_float_p]),
    "gmd_read_nbflag": (ctypes.c_int, [ctypes.c_void_p, c_int_p]),
    "gmd_read_nblist": (ctypes.c_int, [ctypes.c_void_p, c_int_p]),
    "gmd_force_rebuild": (ctypes.c_int, [ctypes.c_void_p]),
    "gmd_set_reorder_interval": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int]),
    "gmd_reorder_stats": (ctypes.c_int, [ctypes.c_void_p, c_int_p, ctypes.POINTER(ctypes.c_longlong)]),
    "gmd_copy_probe": (ctypes.c_int, [ctypes.c_ulonglong, ctypes.c_int, c_float_p]),
    "gmd_fma_probe": (ctypes.c_int, [ctypes.c_int, c_float_p]),
    "gmd_get_thermostat": (ctypes.c_int, [ctypes.c_void_p, c_float_p]),
    "gmd_set_thermostat": (ctypes.c_int, [ctypes.c_void_p, c_float_p]),
    "gmd_get_npt_state": (ctypes.c_int, [ctypes.c_void_p, c_float_p]),
    "gmd_set_npt_state": (ctypes.c_int, [ctypes.c_void_p, c_float_p]),
    "gmd_read_scalar_output": (ctypes.c_int, [ctypes.c_void_p, c_float_p]),
    "gmd_read_conf_output": (ctypes.c_int, [ctypes.c_void_p, c_float_p]),
    "gmd_rdf_create": (ctypes.c_int, [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_void_p)]),
    "gmd_rdf_destroy": (ctypes.c_int, [ctypes.c_void_p]),
    "gmd_rdf_compute_ctx": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, c_int_p, c_u64_p]),
    "gmd_rdf_launch_ctx": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, c_int_p]),
    "gmd_rdf_collect": (ctypes.c_int, [ctypes.c_void_p, c_u64_p]),
    "gmd_rdf_compute_host": (ctypes.c_int, [ctypes.c_void_p, c_float_p, c_int_p, c_float_p, c_u64_p]),
    "gmd_rdf_compute_host_noalloc": (ctypes.c_int, [ctypes.c_int, ctypes.c_int, ctypes.c_int, c_float_p, c_int_p,
                                                    c_float_p, c_u64_p]),
    "gmd_batch_create": (ctypes.c_int, [ctypes.POINTER(GmdDesc), ctypes.c_int, c_int_p, ctypes.c_int,
                                        ctypes.POINTER(ctypes.c_void_p)]),
    "gmd_batch_destroy": (ctypes.c_int, [ctypes.c_void_p]),
    "gmd_batch_size": (ctypes.c_int, [ctypes.c_void_p, c_int_p, c_int_p]),
    "gmd_batch_context": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, ctypes.POINTER(ctypes.c_void_p)]),
    "gmd_batch_run": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_float, ctypes.c_int]),
    "gmd_batch_fetch": (ctypes.c_int, [ctypes.c_void_p]),
    "gmd_batch_last_run_ms": (ctypes.c_int, [ctypes.c_void_p, c_float_p]),
    "gmd_adj_create": (ctypes.c_int, [ctypes.POINTER(GmdAdjDesc), c_int_p, c_float_p, ctypes.POINTER(ctypes.c_void_p)]),
    "gmd_adj_destroy": (ctypes.c_int, [ctypes.c_void_p]),
    "gmd_adj_forward": (ctypes.c_int, [ctypes.c_void_p, c_float_p, c_float_p, c_float_p, c_double_p, c_float_p,
                                       c_float_p]),
    "gmd_adj_backward": (ctypes.c_int, [ctypes.c_void_p, c_double_p, c_double_p, c_float_p, c_float_p]),
    "gmd_adj_last_ms": (ctypes.c_int, [ctypes.c_void_p, c_float_p, c_float_p]),
    "gmd_adj_use_checkpoints": (ctypes.c_int, [ctypes.c_void_p]),
}

BATCH_DRIVER = {"persistent": 0, "graph": 1}

_lib = None
_lock = threading.Lock()


class NativeError(RuntimeError):
    """A call into libgamdpy_amd.so failed (message from gmd_last_error)."""


def library_path():
    return LIB_PATH


def load():
    """Load libgamdpy_amd.so (once) and attach the signatures; raises if absent."""
    global _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(LIB_PATH):
            raise NativeError(
                f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; g.build()'` "
                "or `python -m gamdpy_amd._build` (there is no CPU fallback)")
        lib = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in _SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        if lib.gmd_abi_version() != ABI_VERSION:
            raise NativeError(f"libgamdpy_amd ABI {lib.gmd_abi_version()} != binding ABI {ABI_VERSION}")
        if lib.gmd_desc_size() != ctypes.sizeof(GmdDesc):
            raise NativeError(f"gmd_desc size mismatch: library {lib.gmd_desc_size()}, binding {ctypes.sizeof(GmdDesc)}")
        _lib = lib
        return lib


def check(rc, what=""):
    if rc != 0:
        msg = _lib.gmd_last_error().decode(errors="replace") if _lib is not None else "library not loaded"
        raise NativeError(f"{what}: {msg}" if what else msg)


def fptr(a):
    return a.ctypes.data_as(c_float_p) if a is not None else None


def iptr(a):
    return a.ctypes.data_as(c_int_p) if a is not None else None


def u64ptr(a):
    return a.ctypes.data_as(c_u64_p)


_device_info = None


def device_info():
    """Compute units, wavefront size and name of the current HIP device."""
    global _device_info
    if _device_info is None:
        lib = load()
        info = GmdDeviceInfo()
        check(lib.gmd_get_device_info(ctypes.byref(info)), "gmd_get_device_info")
        _device_info = {"compute_units": info.compute_units, "wavefront_size": info.wavefront_size,
                        "max_threads_per_block": info.max_threads_per_block, "total_mem": info.total_mem,
                        "name": info.name.decode(), "arch": info.arch.decode()}
    return _device_info


def copy_probe(nbytes, reps=3):
    """Mean milliseconds of a plain device copy of nbytes (read nbytes, write
    nbytes) over reps launches."""
    ms = ctypes.c_float()
    check(load().gmd_copy_probe(int(nbytes), int(reps), ctypes.byref(ms)), "gmd_copy_probe")
    return float(ms.value)


def fma_probe(iters=4096):
    """Achieved FP32 TFLOP/s of independent FMA chains (no packed FP32)."""
    tf = ctypes.c_float()
    check(load().gmd_fma_probe(int(iters), ctypes.byref(tf)), "gmd_fma_probe")
    return float(tf.value)


def fill_desc(d, desc_fields, params, exclusions=None):
    """Fill a GmdDesc from a dict of field values; returns the arrays that the
    descriptor points to (keep them alive while the descriptor is used).
    'bonds' ((nbonds, 3) int) and 'bond_params' ((nbond_types, 2) float) set
    the bond fields."""
    params = np.ascontiguousarray(params, dtype=np.float32)
    excl = None if exclusions is None else np.ascontiguousarray(exclusions, dtype=np.int32)
    d.abi_version = ABI_VERSION
    bonds = bpar = None
    for k, v in desc_fields.items():
        if k == "bonds":
            bonds = np.ascontiguousarray(v, dtype=np.int32).reshape(-1, 3)
            d.nbonds = bonds.shape[0]
            d.bonds = iptr(bonds)
        elif k == "bond_params":
            bpar = np.ascontiguousarray(v, dtype=np.float32).reshape(-1, 2)
            d.nbond_types = bpar.shape[0]
            d.bond_params = fptr(bpar)
        elif k == "box":
            d.box = (ctypes.c_float * 3)(*[float(x) for x in v])
        elif k == "tparams":
            d.tparams = (ctypes.c_float * 4)(*[float(x) for x in v])
        elif k == "pparams":
            d.pparams = (ctypes.c_float * 4)(*[float(x) for x in v])
        elif k == "pair_exps":
            d.pair_exps = (ctypes.c_float * 2)(*[float(x) for x in v])
        elif k in ("term_kind", "term_first"):
            setattr(d, k, (ctypes.c_int * 2)(*[int(x) for x in v]))
        elif k == "term_exps":
            d.term_exps = (ctypes.c_float * 4)(*[float(x) for x in v])
        else:
            setattr(d, k, v)
    d.params = fptr(params)
    if excl is not None:
        d.exclusions = iptr(excl)
        d.exclusions_cols = excl.shape[1]
    return params, excl, bonds, bpar


class Context:
    """Owns one gmd_ctx: the device state of one Simulation (or Evaluator).
    A replica of a Batch is a borrowed context (``Context.borrowed``): the
    batch owns it and runs it."""

    def __init__(self, desc_fields, params, exclusions=None):
        self.lib = load()
        d = GmdDesc()
        self._keep = fill_desc(d, desc_fields, params, exclusions)
        self._init_fields(d)
        self._owner = None
        h = ctypes.c_void_p()
        check(self.lib.gmd_create(ctypes.byref(d), ctypes.byref(h)), "gmd_create")
        self.h = h

    def _init_fields(self, d):
        self.desc = d
        self.N = d.N
        self.nscalars = d.nscalars
        self.max_nbs = d.max_nbs
        self._all_columns = {d.sid_u, d.sid_w, d.sid_lap, d.sid_k, d.sid_fsq, d.sid_m} >= set(range(d.nscalars))
        self.saves_per_block = d.scalar_saves_per_block
        self.conf_saves_per_block = d.conf_saves_per_block

    @classmethod
    def borrowed(cls, owner, handle, desc):
        self = cls.__new__(cls)
        self.lib = load()
        self._init_fields(desc)
        self._owner = owner
        self.h = handle
        return self

    def close(self):
        if self._owner is not None:
            self.h = None
            return
        if getattr(self, "h", None) is not None and self.h.value:
            self.lib.gmd_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def upload(self, r=None, v=None, f=None, scalars=None, ptype=None, r_im=None):
        arrs = [None if a is None else np.ascontiguousarray(a, dtype=dt)
                for a, dt in ((r, np.float32), (v, np.float32), (f, np.float32), (scalars, np.float32),
                              (ptype, np.int32), (r_im, np.int32))]
        check(self.lib.gmd_upload(self.h, fptr(arrs[0]), fptr(arrs[1]), fptr(arrs[2]), fptr(arrs[3]),
                                  iptr(arrs[4]), iptr(arrs[5])), "gmd_upload")

    def download(self, vectors=None):
        """(r, v, f, scalars, ptype, r_im) on the host; vectors: three
        C-contiguous (N, 3) float32 arrays to fill with r, v and f instead of
        new ones."""
        N = self.N
        r, v, f = vectors if vectors is not None else (np.empty((N, 3), np.float32) for _ in range(3))
        # (a scalar column without a device array is left as it is: zero)
        sc = (np.empty if self._all_columns else np.zeros)((N, self.nscalars), np.float32)
        pt = np.empty(N, np.int32)
        im = np.empty((N, 3), np.int32)
        check(self.lib.gmd_download(self.h, fptr(r), fptr(v), fptr(f), fptr(sc), iptr(pt), iptr(im)), "gmd_download")
        return r, v, f, sc, pt, im

    def run(self, time_zero, steps):
        check(self.lib.gmd_run(self.h, ctypes.c_float(np.float32(time_zero)), int(steps)), "gmd_run")

    def evaluate(self):
        check(self.lib.gmd_evaluate(self.h), "gmd_evaluate")

    def last_run_ms(self):
        x = ctypes.c_float()
        check(self.lib.gmd_last_run_ms(self.h, ctypes.byref(x)), "gmd_last_run_ms")
        return float(x.value)

    def profile_steps(self, time_zero, steps):
        """Run ``steps`` steps with hipEvents around every kernel; returns the mean
        (step kernel ms, step-tail kernel ms)."""
        a, b = ctypes.c_float(), ctypes.c_float()
        check(self.lib.gmd_profile_steps(self.h, ctypes.c_float(np.float32(time_zero)), int(steps), ctypes.byref(a),
                                         ctypes.byref(b)), "gmd_profile_steps")
        return float(a.value), float(b.value)

    def nbflag(self):
        a = np.zeros(3, np.int32)
        check(self.lib.gmd_read_nbflag(self.h, iptr(a)), "gmd_read_nbflag")
        return a

    def nblist(self):
        a = np.zeros((self.N, self.max_nbs + 1), np.int32)
        check(self.lib.gmd_read_nblist(self.h, iptr(a)), "gmd_read_nblist")
        return a

    def reorder_stats(self):
        """(renumbered now, renumberings so far)"""
        p, n = ctypes.c_int(), ctypes.c_longlong()
        check(self.lib.gmd_reorder_stats(self.h, ctypes.byref(p), ctypes.byref(n)), "gmd_reorder_stats")
        return bool(p.value), int(n.value)

    def set_reorder_interval(self, steps):
        check(self.lib.gmd_set_reorder_interval(self.h, int(steps)), "gmd_set_reorder_interval")

    def force_rebuild(self):
        check(self.lib.gmd_force_rebuild(self.h), "gmd_force_rebuild")

    def get_thermostat(self):
        a = np.zeros(2, np.float32)
        check(self.lib.gmd_get_thermostat(self.h, fptr(a)), "gmd_get_thermostat")
        return a

    def set_thermostat(self, state):
        a = np.ascontiguousarray(state, dtype=np.float32)
        check(self.lib.gmd_set_thermostat(self.h, fptr(a)), "gmd_set_thermostat")

    def get_npt_state(self):
        """[p_xi/Q, p_eps/W, volume, Lx, Ly, Lz] of an NPT_Atomic context."""
        a = np.zeros(6, np.float32)
        check(self.lib.gmd_get_npt_state(self.h, fptr(a)), "gmd_get_npt_state")
        return a

    def current_box(self):
        """The box lengths after the last run when the integrator changes
        them (NPT_Atomic), else None."""
        if self.desc.integrator != INTEGRATOR["NPT_Atomic"]:
            return None
        return self.get_npt_state()[3:6].copy()

    def set_npt_state(self, state):
        a = np.ascontiguousarray(state, dtype=np.float32)
        if a.shape != (6,):
            raise ValueError("the NPT state is [p_xi/Q, p_eps/W, volume, Lx, Ly, Lz]")
        check(self.lib.gmd_set_npt_state(self.h, fptr(a)), "gmd_set_npt_state")

    def scalar_output(self):
        a = np.zeros((self.saves_per_block, len(SAVE_COLUMNS)), np.float32)
        check(self.lib.gmd_read_scalar_output(self.h, fptr(a)), "gmd_read_scalar_output")
        return a

    def conf_output(self):
        """The ConfigurationSaver array of the last block, (saves, 2, N, 3)
        float32 (r, r_im), cleared on the device afterwards."""
        a = np.zeros((self.conf_saves_per_block, 2, self.N, 3), np.float32)
        check(self.lib.gmd_read_conf_output(self.h, fptr(a)), "gmd_read_conf_output")
        return a


class Batch:
    """Owns one gmd_batch: independent replicas advanced by one launch per run
    (driver 'persistent') or one launch per step in a hipGraph ('graph').
    ``replicas`` is a list of (desc_fields, params, exclusions)."""

    def __init__(self, replicas, blocks=None, driver="persistent"):
        self.lib = load()
        n = len(replicas)
        descs = (GmdDesc * n)()
        self._keep = []
        for k, (fields, params, excl) in enumerate(replicas):
            self._keep.append(fill_desc(descs[k], fields, params, excl))
        self._descs = descs
        blk = None if blocks is None else np.ascontiguousarray(blocks, dtype=np.int32)
        if blk is not None and blk.shape != (n,):
            raise ValueError(f"blocks must hold one count per replica ({n})")
        h = ctypes.c_void_p()
        check(self.lib.gmd_batch_create(descs, n, iptr(blk), BATCH_DRIVER[driver], ctypes.byref(h)),
              "gmd_batch_create")
        self.h = h
        self.driver = driver
        self.contexts = []
        for k in range(n):
            c = ctypes.c_void_p()
            check(self.lib.gmd_batch_context(self.h, k, ctypes.byref(c)), "gmd_batch_context")
            self.contexts.append(Context.borrowed(self, c, descs[k]))

    def size(self):
        n, g = ctypes.c_int(), ctypes.c_int()
        check(self.lib.gmd_batch_size(self.h, ctypes.byref(n), ctypes.byref(g)), "gmd_batch_size")
        return n.value, g.value

    def run(self, time_zero, steps):
        check(self.lib.gmd_batch_run(self.h, ctypes.c_float(np.float32(time_zero)), int(steps)), "gmd_batch_run")

    def fetch(self):
        """Bring every replica's state to the host in one go, for the
        downloads that follow."""
        check(self.lib.gmd_batch_fetch(self.h), "gmd_batch_fetch")

    def last_run_ms(self):
        x = ctypes.c_float()
        check(self.lib.gmd_batch_last_run_ms(self.h, ctypes.byref(x)), "gmd_batch_last_run_ms")
        return float(x.value)

    def close(self):
        if getattr(self, "h", None) is not None and self.h.value:
            for c in self.contexts:
                c.h = None
            self.lib.gmd_batch_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class RdfHandle:
    """Owns one gmd_rdf (radial-distribution histogram kernel)."""

    def __init__(self, N, ntypes, bins):
        self.lib = load()
        self.N, self.ntypes, self.bins = int(N), int(ntypes), int(bins)
        h = ctypes.c_void_p()
        check(self.lib.gmd_rdf_create(self.N, self.ntypes, self.bins, ctypes.byref(h)), "gmd_rdf_create")
        self.h = h

    def close(self):
        if getattr(self, "h", None) is not None and self.h.value:
            self.lib.gmd_rdf_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def compute_ctx(self, ctx, ptype=None):
        out = np.zeros((self.ntypes, self.ntypes, self.bins), np.uint64)
        pt = None if ptype is None else np.ascontiguousarray(ptype, dtype=np.int32)
        check(self.lib.gmd_rdf_compute_ctx(self.h, ctx.h, iptr(pt), u64ptr(out)), "gmd_rdf_compute_ctx")
        return out

    def launch_ctx(self, ctx, ptype=None):
        """Start an update from the context's current positions; returns at once."""
        pt = None if ptype is None else np.ascontiguousarray(ptype, dtype=np.int32)
        self._pt = pt   # kept alive until the call returns (the library copies it)
        check(self.lib.gmd_rdf_launch_ctx(self.h, ctx.h, iptr(pt)), "gmd_rdf_launch_ctx")

    def collect(self):
        """Counts of the launched update (waits for it)."""
        out = np.zeros((self.ntypes, self.ntypes, self.bins), np.uint64)
        check(self.lib.gmd_rdf_collect(self.h, u64ptr(out)), "gmd_rdf_collect")
        return out

    def compute_host(self, r, ptype, box):
        out = np.zeros((self.ntypes, self.ntypes, self.bins), np.uint64)
        r = np.ascontiguousarray(r, dtype=np.float32)
        pt = np.ascontiguousarray(ptype, dtype=np.int32)
        bx = np.ascontiguousarray(box, dtype=np.float32)
        check(self.lib.gmd_rdf_compute_host(self.h, fptr(r), iptr(pt), fptr(bx), u64ptr(out)), "gmd_rdf_compute_host")
        return out


def rdf_counts_noalloc(r, ptype, box, ntypes, bins):
    """Ordered-pair RDF counts (ntypes, ntypes, bins) of host positions through
    gmd_rdf_compute_host_noalloc (no device allocation; N <= 65536 and
    ntypes**2 * bins <= 4096)."""
    lib = load()
    r = np.ascontiguousarray(r, dtype=np.float32)
    pt = np.ascontiguousarray(ptype, dtype=np.int32)
    bx = np.ascontiguousarray(box, dtype=np.float32)
    out = np.zeros((ntypes, ntypes, bins), np.uint64)
    check(lib.gmd_rdf_compute_host_noalloc(int(r.shape[0]), int(ntypes), int(bins), fptr(r), iptr(pt), fptr(bx),
                                           u64ptr(out)), "gmd_rdf_compute_host_noalloc")
    return out


def header_functions(path=HEADER_PATH):
    """Names of the gmd_* functions declared in include/gamdpy_amd.h."""
    import re
    txt = open(path).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(gmd_[a-z0-9_]+)\s*\(", txt)))
