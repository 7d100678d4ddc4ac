"""Python handle on the C ABI of libmvd_rhs.so (include/mvd_rhs.h).

Device arrays are torch tensors on the GPU (float64, contiguous); torch is used only to
own device memory and to name the stream. Every compute call goes through the HIP
library; if the library is missing, loading fails loudly.

Load by path (the package directory name is not a Python identifier):
    spec = importlib.util.spec_from_file_location("mvd_pyapi", ".../pyapi.py")
"""
import ctypes as C
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libmvd_rhs.so")
TABLES_PATH = os.path.join(HERE, "data", "primordial_tables.f64")
HEADER_PATH = os.path.join(os.path.dirname(HERE), "include", "mvd_rhs.h")
ARKODE_LIB_PATH = os.path.join(HERE, "libmvd_arkode.so")
ARKODE_HEADER_PATH = os.path.join(os.path.dirname(HERE), "include", "mvd_arkode.h")

MVD_SUCCESS, MVD_ILLEGAL_STATE, MVD_BAD_ARGUMENT = 0, -1, -2
MVD_DEVICE_ERROR, MVD_UNSUPPORTED, MVD_NOT_READY = -3, -4, -5
BC_PERIODIC, BC_NEUMANN, BC_DIRICHLET, BC_REFLECTING = 0, 1, 2, 3


class Params(C.Structure):
    _fields_ = [("nx", C.c_long), ("ny", C.c_long), ("nz", C.c_long), ("nchem", C.c_int),
                ("bc", C.c_int * 6), ("gamma", C.c_double),
                ("xl", C.c_double), ("xr", C.c_double), ("yl", C.c_double),
                ("yr", C.c_double), ("zl", C.c_double), ("zr", C.c_double),
                ("cfl", C.c_double), ("mass_units", C.c_double),
                ("length_units", C.c_double), ("time_units", C.c_double)]


DIRK_MAXSTAGE = 7


class DirkOpts(C.Structure):
    """mvd_dirk_opts: SDIRK or ESDIRK table (row-major 7x7 A) and Newton controls."""
    _fields_ = [("nstage", C.c_int), ("A", C.c_double * 49), ("c", C.c_double * 7),
                ("rtol", C.c_double), ("atol", C.c_double), ("newton_tol", C.c_double),
                ("max_iters", C.c_int), ("max_setups", C.c_int), ("rhs_scale", C.c_double),
                ("max_halvings", C.c_int), ("max_steps_between_setups", C.c_int)]


class ArkTable(C.Structure):
    """mvd_ark_table: explicit / diagonally implicit IMEX pair, up to 8 stages (8x8)."""
    _fields_ = [("stages", C.c_int), ("Ae", C.c_double * 64), ("Ai", C.c_double * 64),
                ("b", C.c_double * 8), ("c", C.c_double * 8)]


class ErkTable(C.Structure):
    """mvd_erk_table: explicit Butcher table, up to 6 stages (row-major 6x6 A)."""
    _fields_ = [("stages", C.c_int), ("A", C.c_double * 36), ("b", C.c_double * 6),
                ("c", C.c_double * 6)]


class DirkStats(C.Structure):
    _fields_ = [("newton_iters", C.c_long), ("max_cell_iters", C.c_int),
                ("failed_cells", C.c_long), ("setups", C.c_long), ("hist", C.c_long * 16),
                ("ms", C.c_double)]

    def as_dict(self):
        return {"newton_iters": self.newton_iters, "max_cell_iters": self.max_cell_iters,
                "failed_cells": self.failed_cells, "setups": self.setups,
                "hist": list(self.hist), "ms": self.ms}


_P = C.POINTER(C.c_double)
_PP = C.POINTER(_P)
_lib = None


def lib():
    """Load libmvd_rhs.so and declare the ABI; raises if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(f"{LIB_PATH} missing: run `python sundials-manyvector-demo_amd/build.py`")
    L = C.CDLL(LIB_PATH)
    vp = C.c_void_p
    sig = {
        "mvd_create": ([C.POINTER(Params), vp, C.POINTER(vp)], C.c_int),
        "mvd_destroy": ([vp], None),
        "mvd_set_stream": ([vp, vp], C.c_int),
        "mvd_fe": ([vp, C.c_double, _PP, _PP], C.c_int),
        "mvd_fe_plain": ([vp, C.c_double, _PP, _PP], C.c_int),
        "mvd_fe_async": ([vp, C.c_double, _PP, _PP], C.c_int),
        "mvd_last_state_flags": ([vp], C.c_int),
        "mvd_fe_vjp": ([vp, C.c_double, _PP, _PP, _PP], C.c_int),
        "mvd_max_wave_speed": ([vp, _PP, _P], C.c_int),
        "mvd_stability": ([vp, _PP, C.c_double, _P], C.c_int),
        "mvd_fslow": ([vp, C.c_double, _PP, _PP], C.c_int),
        "mvd_profile": ([vp, C.c_int], C.c_int),
        "mvd_profile_read": ([vp, _P, C.POINTER(C.c_long), C.c_int], C.c_int),
        "mvd_chem_setup": ([vp, _P, C.c_long, C.c_double], C.c_int),
        "mvd_chem_prepare": ([vp, _P], C.c_int),
        "mvd_chem_apply_scaling": ([vp, _P], C.c_int),
        "mvd_chem_unapply_scaling": ([vp, _P], C.c_int),
        "mvd_chem_rhs": ([vp, C.c_double, _P, _P], C.c_int),
        "mvd_chem_jac": ([vp, C.c_double, _P, _P], C.c_int),
        "mvd_chem_rhs_scaled": ([vp, C.c_double, C.c_double, _P, _P], C.c_int),
        "mvd_chem_jac_scaled": ([vp, C.c_double, C.c_double, _P, _P], C.c_int),
        "mvd_chem_lsetup_matrix": ([vp, _P], C.c_int),
        "mvd_nvec_const": ([vp, C.c_double, _P, C.c_long], C.c_int),
        "mvd_nvec_axpy_steps": ([vp, C.c_int, C.c_double, _P, _P, C.c_long], C.c_int),
        "mvd_mri_fast_steps": ([C.c_int, C.c_double, C.c_double], C.c_int),
        "mvd_postprocess_step": ([vp, C.c_double, _PP], C.c_int),
        "mvd_chem_state": ([vp, C.c_int], _P),
        "mvd_chem_lsetup": ([vp, C.c_double, _P], C.c_int),
        "mvd_nvec_linear_combination": ([vp, C.c_int, _P, C.POINTER(_P), _P, C.c_long],
                                        C.c_int),
        "mvd_nvec_wrms_norm": ([vp, C.c_int, C.POINTER(_P), C.POINTER(_P),
                                C.POINTER(C.c_long), C.POINTER(C.c_double)], C.c_int),
        "mvd_erk_bs3": ([C.POINTER(ErkTable)], C.c_int),
        "mvd_erk_evolve": ([vp, C.POINTER(ErkTable), C.c_double, C.c_double, C.c_int,
                           C.POINTER(_P)], C.c_int),
        "mvd_chem_lsolve": ([vp, _P, _P], C.c_int),
        "mvd_chem_vjp": ([vp, C.c_double, _P, _P, _P, _P], C.c_int),
        "mvd_chem_temperature_check": ([vp, _P, _P, C.POINTER(C.c_long)], C.c_int),
        "mvd_exchange": ([vp, _PP, _PP], C.c_int),
        "mvd_pack1d": ([vp, _PP, C.c_int, C.c_long, C.c_void_p, _P], C.c_int),
        "mvd_dirk_sdirk3": ([C.POINTER(DirkOpts)], C.c_int),
        "mvd_dirk_ark437": ([C.POINTER(DirkOpts)], C.c_int),
        "mvd_chem_dirk_step": ([vp, C.c_double, C.c_double, C.POINTER(DirkOpts), _P, C.c_int,
                                C.POINTER(DirkStats)], C.c_int),
        "mvd_chem_dirk_tune": ([vp, C.c_double, C.POINTER(DirkOpts), _P, _P], C.c_int),
        "mvd_chem_dirk_step_noalloc": ([vp, C.c_double, C.c_double, C.POINTER(DirkOpts), _P,
                                        C.POINTER(DirkStats)], C.c_int),
        "mvd_chem_dirk_set_shape": ([vp, C.c_int, C.c_int], C.c_int),
        "mvd_chem_dirk_fit_block": ([C.c_int, C.c_int, C.c_long, C.c_long], C.c_int),
        "mvd_chem_dirk_get_shape": ([vp, C.POINTER(C.c_int), C.POINTER(C.c_int)], C.c_int),
        "mvd_chem_dirk_step_forced": ([vp, C.c_double, C.c_double, C.POINTER(DirkOpts), _P, _P,
                                       C.POINTER(DirkStats)], C.c_int),
        "mvd_chem_dirk_steps": ([vp, C.c_double, C.c_double, C.c_int, C.POINTER(DirkOpts), _P,
                                 _P, C.POINTER(DirkStats)], C.c_int),
        "mvd_mri_evolve": ([vp, C.c_double, C.c_double, C.c_int, C.c_double,
                            C.POINTER(DirkOpts), C.c_int, C.POINTER(_P)], C.c_int),
        "mvd_ark_ark324": ([C.POINTER(ArkTable)], C.c_int),
        "mvd_ark_ark437": ([C.POINTER(ArkTable)], C.c_int),
        "mvd_imex_evolve": ([vp, C.c_double, C.c_double, C.c_int, C.POINTER(ArkTable),
                             C.POINTER(DirkOpts), C.c_int, C.POINTER(_P)], C.c_int),
        "mvd_chem_dirk_adjoint": ([vp, C.c_double, C.c_double, C.c_int, C.c_int,
                                   C.POINTER(DirkOpts), _P, _P, _P], C.c_int),
    }
    for name, (args, res) in sig.items():
        fn = getattr(L, name)
        fn.argtypes = args
        fn.restype = res
    _lib = L
    return L


def exported_symbols_declared(header=HEADER_PATH):
    """Names declared in a header of include/ (for the ABI completeness tests)."""
    import re
    txt = open(header).read()
    return sorted(set(re.findall(r"\b(mvd_[A-Za-z0-9_]+)\s*\(", txt)))


class ArkodeData(C.Structure):
    """mvd_arkode_data: user data of the ARKODE callbacks (include/mvd_arkode.h)."""
    _fields_ = [("ctx", C.c_void_p), ("time_units", C.c_double), ("stepper", C.c_void_p),
                ("disable_forcing", C.c_int), ("fast", DirkOpts), ("hmax_fast", C.c_double),
                ("tcur", C.c_double), ("fast_steps", C.c_long), ("failed_cells", C.c_long)]


_arkode = None


def arkode_lib():
    """Load libmvd_arkode.so and declare its functions. Its SUNDIALS symbols must already be
    resolvable in the process (SUNDIALS, or a stand-in, loaded with RTLD_GLOBAL)."""
    global _arkode
    if _arkode is not None:
        return _arkode
    lib()
    if not os.path.exists(ARKODE_LIB_PATH):
        raise RuntimeError(f"{ARKODE_LIB_PATH} missing: run `python sundials-manyvector-demo_amd/build.py`")
    L = C.CDLL(ARKODE_LIB_PATH)
    vp, d = C.c_void_p, C.c_double
    rhs = ([d, vp, vp, vp], C.c_int)
    jac = ([d, vp, vp, vp, vp, vp, vp, vp], C.c_int)
    sig = {
        "mvd_arkode_fEuler": rhs, "mvd_arkode_fslow": rhs, "mvd_arkode_ffast": rhs,
        "mvd_arkode_fimpl": rhs, "mvd_arkode_frhs": rhs,
        "mvd_arkode_stability": ([vp, d, C.POINTER(d), vp], C.c_int),
        "mvd_arkode_Jfast": jac, "mvd_arkode_Jimpl": jac, "mvd_arkode_Jrhs": jac,
        "mvd_arkode_postprocess": ([d, vp, vp], C.c_int),
        "mvd_SUNLinSol_RankLocalLS": ([vp, C.c_long, C.POINTER(ArkodeData), vp], vp),
        "mvd_inner_evolve": ([vp, d, d, vp], C.c_int),
        "mvd_inner_fullrhs": ([vp, d, vp, vp, C.c_int], C.c_int),
        "mvd_inner_reset": ([vp, d, vp], C.c_int),
        "mvd_inner_stepper_create": ([vp, C.POINTER(ArkodeData), C.POINTER(vp)], C.c_int),
    }
    for name, (args, res) in sig.items():
        fn = getattr(L, name)
        fn.argtypes = args
        fn.restype = res
    _arkode = L
    return L


# ---------------------------------------------------------------------------------------
# solution output / restart input (libmvd_io.so, include/mvd_io.h)
# ---------------------------------------------------------------------------------------
IO_LIB_PATH = os.path.join(HERE, "libmvd_io.so")
IO_HEADER_PATH = os.path.join(os.path.dirname(HERE), "include", "mvd_io.h")
MVD_IO_ERROR, MVD_IO_MISMATCH = -6, -7


class RunOptions(C.Structure):
    """mvd_run_options: the driver/ARKODE options restart_parameters.txt records; defaults
    are ARKODEParameters' (euler3D.hpp:163-168) with the NONE table ids (-1)."""
    _fields_ = [("tf", C.c_double), ("nout", C.c_int), ("showstats", C.c_int),
                ("order", C.c_int), ("dense_order", C.c_int), ("etable", C.c_int),
                ("itable", C.c_int), ("mtable", C.c_int), ("adapt_method", C.c_int),
                ("maxnef", C.c_int), ("mxhnil", C.c_int), ("mxsteps", C.c_int),
                ("safety", C.c_double), ("bias", C.c_double), ("growth", C.c_double),
                ("pq", C.c_int), ("k1", C.c_double), ("k2", C.c_double), ("k3", C.c_double),
                ("etamx1", C.c_double), ("etamxf", C.c_double), ("hmin", C.c_double),
                ("hmax", C.c_double), ("fixedstep", C.c_int), ("htrans", C.c_double),
                ("rtol", C.c_double), ("atol", C.c_double), ("fusedkernels", C.c_int),
                ("localreduce", C.c_int)]

    def __init__(self, **kw):
        d = dict(tf=1.0, nout=10, showstats=0, order=4, dense_order=-1, etable=-1, itable=-1,
                 mtable=-1, mxsteps=5000, rtol=1e-8, atol=1e-12, fusedkernels=1,
                 localreduce=1)
        d.update(kw)
        super().__init__(**d)


_io = None


def io_lib():
    """Load libmvd_io.so and declare its ABI; raises if it has not been built."""
    global _io
    if _io is not None:
        return _io
    if not os.path.exists(IO_LIB_PATH):
        raise RuntimeError(f"{IO_LIB_PATH} missing: run `python sundials-manyvector-demo_amd/build.py`")
    L = C.CDLL(IO_LIB_PATH)
    PR, RO = C.POINTER(Params), C.POINTER(RunOptions)
    L.mvd_write_parameters.argtypes = [C.c_char_p, PR, RO, C.c_double, C.c_double, C.c_int]
    L.mvd_output_solution.argtypes = [C.c_char_p, PR, RO, C.c_double, C.c_double, C.c_int,
                                      _PP, C.c_int]
    L.mvd_read_restart.argtypes = [C.c_char_p, PR, C.c_int, C.POINTER(C.c_double), _PP,
                                   C.c_int]
    for f in (L.mvd_write_parameters, L.mvd_output_solution, L.mvd_read_restart):
        f.restype = C.c_int
    _io = L
    return L


def _field_ptrs(w):
    """(pointer array, on_device) for six float64 arrays (numpy on the host or torch on the
    device; w[5] may be None without species)."""
    import numpy as np
    dev = any(x is not None and not isinstance(x, np.ndarray) for x in w)
    ps = []
    for x in w:
        if x is None:
            ps.append(_P())
        elif isinstance(x, np.ndarray):
            assert not dev and x.dtype == np.float64 and x.flags.c_contiguous
            ps.append(x.ctypes.data_as(_P))
        else:
            ps.append(dptr(x))
    return C.cast((_P * len(ps))(*ps), _PP), int(dev)


def output_solution(directory, params, t, h, iout, w, options=None):
    """output_solution: restart_parameters.txt (when options is given) and
    output-<iout>.hdf5 in directory from w (numpy host arrays or torch device tensors)."""
    pp, dev = _field_ptrs(w)
    rc = io_lib().mvd_output_solution(str(directory).encode(), C.byref(params),
                                      C.byref(options) if options is not None else None,
                                      t, h, iout, pp, dev)
    return _check("mvd_output_solution", rc)


def read_restart(directory, params, restart, w):
    """read_restart into w (overwritten); returns the stored time."""
    pp, dev = _field_ptrs(w)
    t = C.c_double(0.0)
    rc = io_lib().mvd_read_restart(str(directory).encode(), C.byref(params), restart,
                                   C.byref(t), pp, dev)
    _check("mvd_read_restart", rc)
    return t.value


def write_parameters(directory, params, options, t, h, iout):
    rc = io_lib().mvd_write_parameters(str(directory).encode(), C.byref(params),
                                       C.byref(options), t, h, iout)
    return _check("mvd_write_parameters", rc)


def load_tables():
    """The 50 primordial rate / cooling / gamma tables (50 x 1024, the committed blob in the
    reference's read order, data/primordial_tables.json) for mvd_chem_setup."""
    import numpy as np
    return np.fromfile(TABLES_PATH, dtype="<f8").reshape(50, 1024)


def mri_fast_steps(stage, h, hmax):
    """Fast steps of slow stage `stage` (2..4) of mvd_mri_evolve."""
    return lib().mvd_mri_fast_steps(stage, h, hmax)


def dptr(t):
    """Device pointer of a float64 contiguous torch tensor."""
    assert t.dtype.is_floating_point and t.element_size() == 8 and t.is_contiguous()
    return C.cast(C.c_void_p(t.data_ptr()), _P)


def dptrs(ts):
    arr = (_P * len(ts))(*[dptr(t) if t is not None else _P() for t in ts])
    return C.cast(arr, _PP)


class MvdError(RuntimeError):
    def __init__(self, fn, code):
        super().__init__(f"{fn} returned {code}")
        self.code = code


def _check(fn, rc, allow=(MVD_SUCCESS,)):
    if rc not in allow:
        raise MvdError(fn, rc)
    return rc


def bs3():
    t = ErkTable()
    _check("mvd_erk_bs3", lib().mvd_erk_bs3(C.byref(t)))
    return t


def ark324():
    t = ArkTable()
    _check("mvd_ark_ark324", lib().mvd_ark_ark324(C.byref(t)))
    return t


def ark437_pair():
    """ARK4(3)7L[2]SA, the IMEX pair of the reference's IMEX inputs (etable 13, itable 112)."""
    t = ArkTable()
    _check("mvd_ark_ark437", lib().mvd_ark_ark437(C.byref(t)))
    return t


def make_params(nx, ny, nz, nchem=0, bc=(0,) * 6, gamma=1.4, extent=((0, 1), (0, 1), (0, 1)),
                cfl=0.0, units=(1.0, 1.0, 1.0)):
    p = Params()
    p.nx, p.ny, p.nz, p.nchem = nx, ny, nz, nchem
    for i in range(6):
        p.bc[i] = bc[i]
    p.gamma = gamma
    (p.xl, p.xr), (p.yl, p.yr), (p.zl, p.zr) = extent
    p.cfl = cfl
    p.mass_units, p.length_units, p.time_units = units
    return p


class Context:
    """One mvd_context (the hot-path part of EulerData + cvklu_data)."""

    def __init__(self, params, stream=None):
        self.params = params
        h = C.c_void_p()
        _check("mvd_create", lib().mvd_create(C.byref(params), stream, C.byref(h)))
        self.h = h

    def close(self):
        if getattr(self, "h", None):
            lib().mvd_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:   # interpreter shutdown: the library may already be unloaded
            pass

    # fe() family ------------------------------------------------------------------------
    def fe(self, w, wdot, t=0.0, plain=False, allow_illegal=False):
        fn = lib().mvd_fe_plain if plain else lib().mvd_fe
        allow = (MVD_SUCCESS, MVD_ILLEGAL_STATE) if allow_illegal else (MVD_SUCCESS,)
        return _check("mvd_fe", fn(self.h, t, dptrs(w), dptrs(wdot)), allow)

    def exchange(self, w, recv):
        """Fill the six ghost receive buffers (W, E, S, N, B, F; None skips one)."""
        _check("mvd_exchange", lib().mvd_exchange(self.h, dptrs(w), dptrs(recv)))

    def pack1d(self, w, d, ijk, out):
        """Stencils w(c-3..c+2) along d of the cells ijk (int32 device tensor [n][3])."""
        assert ijk.dtype.itemsize == 4 and ijk.is_contiguous()
        n = ijk.numel() // 3
        _check("mvd_pack1d", lib().mvd_pack1d(self.h, dptrs(w), d, n, C.c_void_p(ijk.data_ptr()),
                                              dptr(out)))

    def erk_evolve(self, w, h, nsteps, table=None, t0=0.0, allow_illegal=False):
        """Fixed-step explicit RK of fe() in place on w (default table: Bogacki-Shampine 3)."""
        tab = table if table is not None else bs3()
        allow = (MVD_SUCCESS, MVD_ILLEGAL_STATE) if allow_illegal else (MVD_SUCCESS,)
        return _check("mvd_erk_evolve", lib().mvd_erk_evolve(
            self.h, C.byref(tab), t0, h, int(nsteps), dptrs(w)), allow)

    def linear_combination(self, c, X, z):
        import numpy as np
        cc = np.ascontiguousarray(c, dtype=np.float64)
        xs = (_P * len(X))(*[dptr(x) for x in X])
        _check("mvd_nvec_linear_combination", lib().mvd_nvec_linear_combination(
            self.h, len(X), cc.ctypes.data_as(_P), xs, dptr(z), z.numel()))

    def wrms_norm(self, xs, ws):
        n = len(xs)
        xp = (_P * n)(*[dptr(x) for x in xs])
        wp = (_P * n)(*[dptr(x) for x in ws])
        ln = (C.c_long * n)(*[x.numel() for x in xs])
        out = C.c_double(0.0)
        _check("mvd_nvec_wrms_norm", lib().mvd_nvec_wrms_norm(self.h, n, xp, wp, ln, C.byref(out)))
        return out.value

    def fe_async(self, w, wdot, t=0.0):
        return _check("mvd_fe_async", lib().mvd_fe_async(self.h, t, dptrs(w), dptrs(wdot)))

    def fe_vjp(self, w, v, wbar, t=0.0):
        return _check("mvd_fe_vjp", lib().mvd_fe_vjp(self.h, t, dptrs(w), dptrs(v), dptrs(wbar)))

    def last_state_flags(self):
        return lib().mvd_last_state_flags(self.h)

    def max_wave_speed(self, w):
        a = C.c_double()
        _check("mvd_max_wave_speed", lib().mvd_max_wave_speed(self.h, dptrs(w), C.byref(a)))
        return a.value

    def stability(self, w, t=0.0):
        d = C.c_double()
        _check("mvd_stability", lib().mvd_stability(self.h, dptrs(w), t, C.byref(d)))
        return d.value

    def fslow(self, w, wdot, t=0.0):
        return _check("mvd_fslow", lib().mvd_fslow(self.h, t, dptrs(w), dptrs(wdot)))

    # slots 0 and 1 are unused; slot 2 times the z-face kernels (fluid, then tracers)
    PROFILE_SLOTS = ("unused0", "unused1", "fe_zface_div", "fe_plain_faces", "fe_plain_div",
                     "fe_xyface_div", "fe_box")

    def profile(self, on=True):
        _check("mvd_profile", lib().mvd_profile(self.h, 1 if on else 0))

    def profile_read(self):
        n = len(self.PROFILE_SLOTS)
        ms = (C.c_double * n)()
        cnt = (C.c_long * n)()
        rc = lib().mvd_profile_read(self.h, ms, cnt, n)
        if rc < 0:
            raise MvdError("mvd_profile_read", rc)
        return {name: (ms[i], cnt[i]) for i, name in enumerate(self.PROFILE_SLOTS)}

    # chemistry ---------------------------------------------------------------------------
    def chem_setup(self, tables, ncell, current_z=-1.0):
        import numpy as np
        tab = np.ascontiguousarray(tables, dtype=np.float64).reshape(-1)
        assert tab.size == 50 * 1024
        _check("mvd_chem_setup", lib().mvd_chem_setup(
            self.h, tab.ctypes.data_as(_P), ncell, current_z))
        self.ncell = ncell

    def chem_prepare(self, chem):
        _check("mvd_chem_prepare", lib().mvd_chem_prepare(self.h, dptr(chem)))

    def chem_apply_scaling(self, chem):
        _check("mvd_chem_apply_scaling", lib().mvd_chem_apply_scaling(self.h, dptr(chem)))

    def chem_unapply_scaling(self, chem):
        _check("mvd_chem_unapply_scaling", lib().mvd_chem_unapply_scaling(self.h, dptr(chem)))

    def chem_rhs(self, y, ydot, t=0.0):
        _check("mvd_chem_rhs", lib().mvd_chem_rhs(self.h, t, dptr(y), dptr(ydot)))

    def chem_jac(self, y, J, t=0.0):
        _check("mvd_chem_jac", lib().mvd_chem_jac(self.h, t, dptr(y), dptr(J)))

    def mri_evolve(self, w, h, nslow, hmax_fast, fast_opts, consistent=False, t0=0.0):
        """Multirate evolution (MIS Knoth-Wolke 3 slow, forced batched DIRK fast with steps of
        at most hmax_fast) in place on w; returns the failed fast cell steps (0: all
        converged). consistent: chemistry forcing in the fast stepper's scaled variables."""
        rc = lib().mvd_mri_evolve(self.h, t0, h, int(nslow), hmax_fast, C.byref(fast_opts),
                                  1 if consistent else 0, dptrs(w))
        if rc < 0:
            _check("mvd_mri_evolve", rc)
        return rc

    def imex_evolve(self, w, h, nsteps, newton, table=None, consistent=False, t0=0.0):
        """IMEX ARK evolution (explicit fexpl, implicit chemistry; default table
        ARK3(2)4L[2]SA) in place on w; returns the failed cell solves (0: all converged)."""
        tab = table if table is not None else ark324()
        rc = lib().mvd_imex_evolve(self.h, t0, h, int(nsteps), C.byref(tab), C.byref(newton),
                                   1 if consistent else 0, dptrs(w))
        if rc < 0:
            _check("mvd_imex_evolve", rc)
        return rc

    def dirk_step_forced(self, y, h, force, opts=None, t=0.0):
        o = opts if opts is not None else sdirk3()
        st = DirkStats()
        rc = lib().mvd_chem_dirk_step_forced(self.h, t, h, C.byref(o), dptr(y), dptr(force),
                                             C.byref(st))
        if rc < 0:
            _check("mvd_chem_dirk_step_forced", rc)
        return rc

    def dirk_steps(self, y, h, nsteps, force=None, opts=None, t=0.0):
        """mvd_chem_dirk_steps: nsteps steps of size h per cell in one launch (force
        optional). Returns (failed cell steps, stats)."""
        o = opts if opts is not None else sdirk3()
        st = DirkStats()
        rc = lib().mvd_chem_dirk_steps(self.h, t, h, int(nsteps), C.byref(o), dptr(y),
                                       dptr(force) if force is not None else None,
                                       C.byref(st))
        if rc < 0:
            _check("mvd_chem_dirk_steps", rc)
        return rc, st.as_dict()

    def nvec_axpy_steps(self, nsteps, a, x, y):
        """mvd_nvec_axpy_steps: y = 1 y + a x, nsteps times in turn."""
        _check("mvd_nvec_axpy_steps", lib().mvd_nvec_axpy_steps(self.h, int(nsteps), a,
                                                                dptr(x), dptr(y), y.numel()))

    def dirk_adjoint(self, y, h, nsteps, ckpt_every, lamT, lam0, opts=None, t=0.0):
        """Checkpointed adjoint of nsteps DIRK steps: y advanced in place, lam0 filled with
        (dy_N/dy_0)^T lamT. Returns the number of cells whose forward Newton failed."""
        o = opts if opts is not None else sdirk3()
        rc = lib().mvd_chem_dirk_adjoint(self.h, t, h, int(nsteps), int(ckpt_every), C.byref(o),
                                         dptr(y), dptr(lamT), dptr(lam0))
        if rc < 0:
            _check("mvd_chem_dirk_adjoint", rc)
        return rc

    def chem_lsetup(self, gamma, J):
        """Factor A = I - gamma*J per cell; returns the number of singular blocks (0: ok)."""
        rc = lib().mvd_chem_lsetup(self.h, gamma, dptr(J))
        if rc < 0:
            _check("mvd_chem_lsetup", rc)
        return rc

    def chem_lsolve(self, b, x):
        _check("mvd_chem_lsolve", lib().mvd_chem_lsolve(self.h, dptr(b), dptr(x)))

    def chem_vjp(self, y, v, ybar, ydot=None, t=0.0):
        _check("mvd_chem_vjp", lib().mvd_chem_vjp(
            self.h, t, dptr(y), dptr(v), dptr(ybar), dptr(ydot) if ydot is not None else _P()))

    def temperature_check(self, y, Ts0):
        """Cells whose early-exit device temperature solve differs bitwise from the ten
        Newton steps, from the warm starts Ts0 (device arrays)."""
        bad = C.c_long()
        _check("mvd_chem_temperature_check", lib().mvd_chem_temperature_check(
            self.h, dptr(y), dptr(Ts0), C.byref(bad)))
        return bad.value

    def chem_state(self, which, torch_mod):
        """Copy of a per-cell state array (see mvd_chem_state) as a torch device tensor."""
        names = {"scale": 0, "inv_scale": 1, "Ts": 2, "dTs_ge": 3, "mdensity": 4,
                 "inv_mdensity": 5, "cie_oda": 6, "h2_oda": 7}
        w = names[which]
        n = self.ncell * (10 if w in (0, 1) else 1)
        ptr = lib().mvd_chem_state(self.h, w)
        if not ptr:
            raise MvdError("mvd_chem_state", MVD_NOT_READY)
        out = torch_mod.empty(n, dtype=torch_mod.float64, device="cuda")
        torch_mod.cuda.synchronize()
        _memcpy_d2d(out.data_ptr(), C.cast(ptr, C.c_void_p).value, n * 8)
        return out


    def chem_state_set(self, which, src):
        """Overwrite a per-cell state array (see chem_state) from a torch device tensor."""
        names = {"scale": 0, "inv_scale": 1, "Ts": 2, "dTs_ge": 3, "mdensity": 4,
                 "inv_mdensity": 5, "cie_oda": 6, "h2_oda": 7}
        w = names[which]
        n = self.ncell * (10 if w in (0, 1) else 1)
        assert src.numel() == n and src.dtype.itemsize == 8 and src.is_contiguous()
        ptr = lib().mvd_chem_state(self.h, w)
        if not ptr:
            raise MvdError("mvd_chem_state", MVD_NOT_READY)
        _memcpy_d2d(C.cast(ptr, C.c_void_p).value, src.data_ptr(), n * 8)

    # implicit chemistry step ------------------------------------------------------------
    def dirk_step(self, y, h, opts=None, plain=False, t=0.0):
        """One SDIRK step of every cell (y scaled, overwritten). Returns (failed, stats)."""
        o = opts if opts is not None else sdirk3()
        st = DirkStats()
        rc = lib().mvd_chem_dirk_step(self.h, t, h, C.byref(o), dptr(y), 1 if plain else 0,
                                      C.byref(st))
        if rc < 0:
            raise MvdError("mvd_chem_dirk_step", rc)
        return rc, st.as_dict()

    def dirk_set_shape(self, block=256, waves=0):
        _check("mvd_chem_dirk_set_shape", lib().mvd_chem_dirk_set_shape(self.h, block, waves))

    def dirk_get_shape(self):
        b, w = C.c_int(), C.c_int()
        _check("mvd_chem_dirk_get_shape", lib().mvd_chem_dirk_get_shape(self.h, C.byref(b),
                                                                        C.byref(w)))
        return b.value, w.value

    def dirk_step_noalloc(self, y, h, opts=None, t=0.0):
        """mvd_chem_dirk_step_noalloc (batched step, no device allocation). Returns (failed,
        stats)."""
        o = opts if opts is not None else sdirk3()
        st = DirkStats()
        rc = lib().mvd_chem_dirk_step_noalloc(self.h, t, h, C.byref(o), dptr(y), C.byref(st))
        if rc < 0:
            raise MvdError("mvd_chem_dirk_step_noalloc", rc)
        return rc, st.as_dict()

    def dirk_tune(self, y, h, opts=None):
        o = opts if opts is not None else sdirk3()
        ms = C.c_double()
        _check("mvd_chem_dirk_tune", lib().mvd_chem_dirk_tune(self.h, h, C.byref(o), dptr(y),
                                                              C.byref(ms)))
        return ms.value


def sdirk3(**kw):
    """Alexander's 3-stage SDIRK with the default Newton controls; keyword overrides."""
    o = DirkOpts()
    _check("mvd_dirk_sdirk3", lib().mvd_dirk_sdirk3(C.byref(o)))
    for k, v in kw.items():
        setattr(o, k, v)
    return o


def ark437(**kw):
    """The ESDIRK part of ARK4(3)7L[2]SA (the reference inputs' implicit table, ARKODE's
    ARK437L2SA_DIRK_7_3_4) with the default Newton controls; keyword overrides."""
    o = DirkOpts()
    _check("mvd_dirk_ark437", lib().mvd_dirk_ark437(C.byref(o)))
    for k, v in kw.items():
        setattr(o, k, v)
    return o


def set_table(o, A, c=None):
    """Puts a square Butcher matrix (up to 7x7, rows as sequences) and its nodes (default:
    the row sums) into DirkOpts o."""
    s = len(A)
    for k in range(DIRK_MAXSTAGE * DIRK_MAXSTAGE):
        o.A[k] = 0.0
    for i in range(s):
        for j in range(s):
            o.A[DIRK_MAXSTAGE * i + j] = float(A[i][j])
    cc = [sum(float(x) for x in A[i]) for i in range(s)] if c is None else list(c)
    for k in range(DIRK_MAXSTAGE):
        o.c[k] = float(cc[k]) if k < s else 0.0
    o.nstage = s
    return o


def _memcpy_d2d(dst, src, nbytes):
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipMemcpy.restype = C.c_int
    rc = hip.hipMemcpy(C.c_void_p(dst), C.c_void_p(src), nbytes, 3)  # hipMemcpyDeviceToDevice
    if rc != 0:
        raise MvdError("hipMemcpy", rc)
