"""ctypes binding of ``libptychotomo_hip.so`` (the C ABI in
``include/ptychotomo_hip.h``).

The shared library is required: importing this module without it raises
``ImportError`` -- there is no CPU fallback anywhere in the package.
"""
import ctypes
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("PTYCHOTOMO_HIP_LIB", os.path.join(HERE, "libptychotomo_hip.so"))

if not os.path.exists(LIB_PATH):
    raise ImportError(
        f"ptychotomo_amd: HIP library not found at {LIB_PATH}; build it with "
        "`python -m ptychotomo_amd.build`")

lib = ctypes.CDLL(LIB_PATH)


def _header_digest():
    import hashlib
    path = os.path.join(HERE, "..", "include", "ptychotomo_hip.h")
    with open(path, "rb") as fh:
        return hashlib.sha256(fh.read()).hexdigest()[:16]


# A library built from another version of the header may take other
# parameter lists than the ones bound below; a call would then pass its
# arguments in the wrong registers (crashing inside the HIP runtime), so it
# is refused here.
lib.pt_header_digest.restype = ctypes.c_char_p
_built = lib.pt_header_digest().decode()
if _built != _header_digest():
    raise ImportError(
        f"ptychotomo_amd: {LIB_PATH} was built from another version of "
        f"include/ptychotomo_hip.h (digest {_built}, header {_header_digest()}); rebuild it "
        "with `python -m ptychotomo_amd.build`")

c_int = ctypes.c_int
c_long = ctypes.c_long
c_float = ctypes.c_float
c_double = ctypes.c_double
vp = ctypes.c_void_p
PT_OK = 0
PT_MODEL = {"gaussian": 0, "poisson": 1}
PT_FILTER = {None: 0, "none": 0, "ramp": 1}
PT_LINES = {"auto": 0, "generic": 1}



class LinesearchArgs(ctypes.Structure):
    """pt_ptycho_linesearch_args (one instance of pt_ptycho_linesearch_group)"""
    _fields_ = [("h", vp), ("f1", vp), ("f2", vp), ("psi", vp), ("dir", vp), ("data", vp),
                ("hh", vp), ("lamd", vp), ("rho", c_double), ("rho_dev", vp), ("gammas", vp),
                ("chunk", c_int), ("coefptycho", c_float), ("coefdata", c_float), ("skip", vp)]


class SweepArgs(ctypes.Structure):
    """pt_ptycho_sweep_args (one instance of pt_ptycho_linesearch_sweep_group)"""
    _fields_ = [("cand_next", vp), ("step", vp), ("w", vp)]


class GradArgs(ctypes.Structure):
    """pt_ptycho_grad_args (one instance of pt_ptycho_grad_group)"""
    _fields_ = [("h", vp), ("grad", vp), ("psi", vp), ("data", vp), ("hh", vp), ("lamd", vp),
                ("rho", c_double), ("rho_dev", vp), ("coefptycho", c_float),
                ("coefdata", c_float)]


_SIGS = {
    "pt_last_error": (ctypes.c_char_p, []),
    "pt_abi_version": (c_int, []),
    "pt_header_digest": (ctypes.c_char_p, []),
    "pt_prof_start": (c_int, [ctypes.c_char_p]),
    "pt_prof_stop": (c_int, [ctypes.POINTER(c_double), ctypes.POINTER(c_long)]),
    "pt_tomo_create": (c_int, [c_int, c_int, c_int, ctypes.POINTER(vp)]),
    "pt_tomo_destroy": (c_int, [vp]),
    "pt_tomo_set_theta": (c_int, [vp, vp, vp]),
    "pt_tomo_fwd": (c_int, [vp, vp, vp, vp]),
    "pt_tomo_adj": (c_int, [vp, vp, vp, vp]),
    "pt_tomo_fwd_scaled": (c_int, [vp, vp, vp, c_float, vp]),
    "pt_tomo_adj_scaled": (c_int, [vp, vp, vp, c_float, vp]),
    "pt_tomo_set_filter": (c_int, [vp, c_int]),
    "pt_tomo_get_tuning": (c_int, [vp, ctypes.POINTER(c_int), ctypes.POINTER(c_int),
                                   ctypes.POINTER(c_int)]),
    "pt_tomo_set_tuning": (c_int, [vp, c_int, c_int, c_int]),
    "pt_tomo_set_line_kernels": (c_int, [vp, c_int]),
    "pt_tomo_get_line_kernels": (c_int, [vp, ctypes.POINTER(c_int)]),
    "pt_ptycho_create": (c_int, [c_int] * 8 + [ctypes.POINTER(vp)]),
    "pt_ptycho_destroy": (c_int, [vp]),
    "pt_ptycho_set_scan_probe": (c_int, [vp, vp, vp, vp]),
    "pt_ptycho_fwd": (c_int, [vp, vp, vp, vp]),
    "pt_ptycho_adj": (c_int, [vp, vp, vp, vp]),
    "pt_ptycho_fwd_scaled": (c_int, [vp, vp, vp, c_float, vp]),
    "pt_ptycho_adj_scaled": (c_int, [vp, vp, vp, c_float, vp]),
    "pt_ptycho_intensity": (c_int, [vp, vp, vp, c_float, c_float, vp]),
    "pt_ptycho_grad": (c_int, [vp, vp, vp, vp, vp, vp, c_double, vp, c_float, c_float, c_int,
                               vp]),
    "pt_ptycho_minf": (c_int, [vp, vp, vp, vp, vp, vp, c_int, c_int, c_float, c_float, c_int,
                               c_int, vp, vp]),
    "pt_ptycho_minf_noalloc": (c_int, [vp, vp, vp, vp, vp, vp, c_int, c_int, c_float, c_float,
                                       c_int, c_int, vp, vp]),
    "pt_ptycho_linesearch_sweep": (c_int, [ctypes.POINTER(LinesearchArgs), vp, vp, vp, c_int, c_int,
                                           c_int, c_int, vp]),
    "pt_ptycho_linesearch_sweep_group": (c_int, [ctypes.POINTER(LinesearchArgs),
                                                 ctypes.POINTER(SweepArgs)] + [c_int] * 5 + [vp]),
    "pt_ptycho_linesearch": (c_int, [vp, vp, vp, vp, vp, vp, vp, vp, c_double, vp, vp, c_int,
                                     c_int, c_float, c_float, c_int, vp, vp]),
    "pt_ptycho_linesearch_group": (c_int, [ctypes.POINTER(LinesearchArgs), c_int, c_int, c_int,
                                           vp]),
    "pt_ptycho_grad_group": (c_int, [ctypes.POINTER(GradArgs), c_int, c_int, vp]),
    "pt_k_dot": (c_int, [vp, vp, vp, c_long, c_int, vp]),
    "pt_k_norm2": (c_int, [vp, vp, c_long, c_int, vp]),
    "pt_k_norm2_lin": (c_int, [vp, vp, vp, c_double, c_double, c_double, c_double, c_long, c_int,
                               vp]),
    "pt_k_lincomb": (c_int, [vp, vp, vp, vp, vp, c_long, c_int, vp]),
    "pt_k_dy_update": (c_int, [vp, vp, vp, c_int, c_long, c_int, vp]),
    "pt_k_dy_reduce": (c_int, [vp, vp, vp, vp, c_long, c_int, vp]),
    "pt_k_reg_fwd": (c_int, [vp, vp, c_int, c_int, c_int, vp]),
    "pt_k_reg_adj": (c_int, [vp, vp, c_int, c_int, c_int, vp]),
    "pt_k_reg_solve": (c_int, [vp, vp, vp, c_double, vp, c_double, c_int, c_int, c_int, vp]),
    "pt_k_exptomo": (c_int, [vp, vp, c_double, c_double, vp, c_long, vp]),
    "pt_k_mlog": (c_int, [vp, vp, c_long, vp]),
    "pt_k_takexi_stats": (c_int, [vp, vp, vp, c_double, vp, c_int, c_int, c_int, c_int, vp]),
    "pt_k_takexi": (c_int, [vp, vp, vp, vp, c_double, c_double, c_double, c_double, c_double,
                            c_double, c_long, vp]),
    "pt_k_takexi_dev": (c_int, [vp, vp, vp, vp, vp, vp, vp, c_double, c_double, c_double,
                                c_double, c_long, vp]),
    "pt_k_tomo_resid": (c_int, [vp, vp, vp, vp, vp, c_double, vp, c_long, vp]),
    "pt_k_reg_grad": (c_int, [vp, vp, vp, vp, c_double, vp, c_int, c_int, c_int, vp]),
    "pt_k_rho_minf": (c_int, [vp, vp, vp, vp, vp, c_double, vp, vp, c_int, c_long, c_int, vp,
                              vp]),
    "pt_k_tomo_minf": (c_int, [vp, vp, vp, vp, vp, vp, c_int, c_long, vp, vp]),
    "pt_k_reg_minf": (c_int, [vp, vp, vp, vp, vp, c_int, c_int, c_int, c_int, vp, vp]),
    "pt_k_dot_diff": (c_int, [vp, vp, vp, vp, c_long, vp]),
    "pt_k_tv_norm": (c_int, [vp, vp, c_long, vp]),
    "pt_k_lincomb3": (c_int, [vp, c_double, c_double, vp, c_double, c_double, vp, c_double,
                              c_double, vp, c_long, vp]),
    "pt_k_axpy_seg": (c_int, [vp, vp, vp, c_long, c_int, vp]),
    "pt_k_max_angle": (c_int, [vp, vp, c_long, vp]),
    "pt_k_intensity": (c_int, [vp, vp, c_float, c_long, vp]),
    "pt_k_dual": (c_int, [vp, vp, vp, vp, c_double, vp, c_int, c_long, vp]),
    "pt_k_dai_yuan": (c_int, [vp, vp, c_int, vp]),
    "pt_k_cg_resid": (c_int, [vp] * 7 + [c_long, vp]),
    "pt_k_cg_reg_grad": (c_int, [vp] * 4 + [c_int, c_int, c_int, vp]),
    "pt_k_split_update": (c_int, [vp] * 6 + [c_double, c_int, c_int, c_int, vp]),
    "pt_k_object_update": (c_int, [vp] * 5 + [c_double, vp, vp, c_long, vp]),
    "pt_k_ls_begin": (c_int, [vp, vp, c_int, c_int, vp]),
    "pt_k_ls_select": (c_int, [vp, vp, vp, vp, vp, vp, vp, c_int, c_int, c_int, c_int, vp]),
    "pt_k_tomo_linesearch": (c_int, [vp] * 10 + [c_long, c_int, c_int, c_int, vp]),
    "pt_k_penalty": (c_int, [vp, vp, vp]),
    "pt_nn_conv3d": (c_int, [vp, vp, vp, vp, c_int, c_int, c_int, c_int, c_int, c_int, vp]),
    "pt_nn_conv3d_wflip": (c_int, [vp, vp, c_int, c_int, vp]),
    "pt_nn_conv3d_wgrad": (c_int, [vp, vp, vp, c_long, vp, vp, vp, c_int, c_int, c_int, c_int,
                                   c_int, vp]),
    "pt_nn_relu_bwd": (c_int, [vp, vp, vp, c_long, vp]),
    "pt_nn_pool": (c_int, [vp, vp, c_int, c_int, c_int, c_int, vp]),
    "pt_nn_pool_bwd": (c_int, [vp, vp, vp, c_int, c_int, c_int, c_int, vp]),
    "pt_nn_up": (c_int, [vp, vp, c_int, c_int, c_int, c_int, c_int, c_int, vp]),
    "pt_nn_up_bwd": (c_int, [vp, vp, c_int, c_int, c_int, c_int, c_int, c_int, vp]),
    "pt_nn_chan_copy": (c_int, [vp, c_int, c_int, vp, c_int, c_int, c_int, c_long, vp]),
    "pt_nn_head": (c_int, [vp, vp, vp, vp, vp, c_long, c_int, c_int, vp]),
    "pt_nn_head_bwd": (c_int, [vp, vp, vp, c_long, vp, vp, vp, c_long, c_int, c_int, vp]),
    "pt_nn_mse": (c_int, [vp, c_int, vp, vp, vp, c_long, vp]),
    "pt_nn_adam": (c_int, [vp, vp, vp, vp, vp, c_long, c_int, c_int, c_float, c_float, c_float,
                           c_float, c_int, vp]),
    "pt_nn_pack_w": (c_int, [vp, vp, c_int, c_int, vp]),
    "pt_nn_to_bf16": (c_int, [vp, vp, c_long, vp]),
    "pt_nn_to_f32": (c_int, [vp, vp, c_long, vp]),
    "pt_nn_mfma_tile": (c_int, [vp, vp, vp, vp]),
    "pt_nn_mfma32_tile": (c_int, [vp, vp, vp, vp]),
}

EXPORTED = sorted(_SIGS)


def _bind():
    for name, (res, args) in _SIGS.items():
        fn = getattr(lib, name, None)
        if fn is None:
            continue
        fn.restype = res
        fn.argtypes = args


_bind()


class PtError(RuntimeError):
    pass


def check(rc, what=""):
    if rc != PT_OK:
        msg = lib.pt_last_error().decode(errors="replace")
        raise PtError(f"{what or 'ptychotomo_hip'} failed ({rc}): {msg}")
    return rc


def call(name, *args):
    """Call a C-ABI function and raise PtError on a non-zero status."""
    return check(getattr(lib, name)(*args), name)


def missing_symbols():
    return [n for n in EXPORTED if getattr(lib, n, None) is None]
