"""ctypes binding of libitomo.so (the C ABI declared in include/itomo.h).

The library is loaded from this package directory; if it is missing the import of any
projector raises :class:`ItomoError` -- there is no CPU fallback.
"""
import ctypes
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libitomo.so")

ITOMO_OK = 0
PROJ = {"dd": 0, "rd": 1, "pd": 2, "ss": 3}
ARITH = {"fast": 0, "ieee": 1}
PENALTY = {None: 0, "huber": 1, "tikhonov": 2, "haar": 3}
DOT_WORK = 3072


class ItomoError(RuntimeError):
    """A libitomo call returned a non-zero status."""


_lib = None

_vp = ctypes.c_void_p
_i = ctypes.c_int
_f = ctypes.c_float
_i64 = ctypes.c_int64

_SIGS = {
    "itomo_version": ([], ctypes.c_char_p),
    "itomo_last_error": ([], ctypes.c_char_p),
    "itomo_radon_dd": ([_vp, _i, _vp, _i, _i, _vp, _vp], _i),
    "itomo_radon_rd": ([_vp, _i, _vp, _i, _i, _vp, _vp], _i),
    "itomo_radon_pd": ([_vp, _i, _vp, _i, _i, _i, _vp, _vp], _i),
    "itomo_radon_ss": ([_vp, _i, _vp, _i, _i, _i, _vp, _vp], _i),
    "itomo_plan_create": ([ctypes.POINTER(_vp), _i, _i, _vp, _i, _i], _i),
    "itomo_plan_create_pd": ([ctypes.POINTER(_vp), _i, _vp, _i, _i, _i], _i),
    "itomo_plan_create_ss": ([ctypes.POINTER(_vp), _i, _vp, _i, _i, _i], _i),
    "itomo_plan_destroy": ([_vp], _i),
    "itomo_plan_trig": ([_vp, _vp, _vp], _i),
    "itomo_plan_set_shapes": ([_vp, _i, _i], _i),
    "itomo_plan_get_shapes": ([_vp, _vp, _vp], _i),
    "itomo_plan_rd_matrix": ([_vp, _i, _vp, _vp], _i),
    "itomo_forward": ([_vp, _vp, _vp, _i, _i, _vp], _i),
    "itomo_back": ([_vp, _vp, _vp, _i, _i, _vp], _i),
    "itomo_sirt_weights": ([_vp, _vp, _vp, _vp], _i),
    "itomo_sirt_forward": ([_vp, _vp, _vp, _vp, _vp, _i, _vp, _vp], _i),
    "itomo_sirt_back": ([_vp, _vp, _vp, _vp, _i, _f, _vp, _vp], _i),
    "itomo_sirt_iterate": ([_vp, _vp, _vp, _vp, _vp, _vp, _i, _f, _vp, _vp], _i),
    "itomo_sirt_iterate_noalloc": ([_vp, _vp, _vp, _vp, _vp, _vp, _i, _f, _vp, _vp], _i),
    "itomo_sirt_constraints": ([_vp, _i, _i, _i, _i, _vp, _vp, _i, _f, _vp, _vp, _vp, _vp], _i),
    "itomo_sirt_residual": ([_vp, _vp, _vp, _i64, _i, _vp, _vp, _vp], _i),
    "itomo_sirt_update": ([_vp, _vp, _vp, _i64, _i, _f, _vp, _vp, _vp], _i),
    "itomo_reciprocal": ([_vp, _vp, _i64, _vp], _i),
    "itomo_mlem_weights": ([_vp, _vp, _vp], _i),
    "itomo_mlem_forward": ([_vp, _vp, _vp, _vp, _i, _vp, _vp], _i),
    "itomo_mlem_back": ([_vp, _vp, _vp, _vp, _i, _vp, _vp], _i),
    "itomo_mlem_iterate": ([_vp, _vp, _vp, _vp, _vp, _i, _vp, _vp], _i),
    "itomo_dot_f64": ([_vp, _vp, _i64, _vp, _vp, _vp], _i),
    "itomo_l1_residual": ([_vp, _vp, _vp, _vp, _vp, _i, _i, _f, _vp, _vp, _vp], _i),
    "itomo_admm_l1_update": ([_vp, _vp, _vp, _i, _i, _f, _f, _vp, _vp, _vp], _i),
    "itomo_penalty": ([_vp, _i, _i, _i, _i, _f, _i, _vp, _vp, _vp], _i),
    "itomo_sobel_magnitude": ([_vp, _i, _i, _i, _vp, _vp], _i),
    "itomo_sps_step": ([_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _f, _f, _i, _vp, _vp], _i),
    "itomo_unet_conv3x3": ([_vp, _i, _i, _i, _i, _vp, _vp, _i, _vp, _i, _vp, _vp], _i),
    "itomo_unet_flip": ([_vp, _i, _i, _vp, _vp], _i),
    "itomo_unet_wgrad": ([_vp, _vp, _i, _i, _i, _i, _i, _vp, _vp, _vp], _i),
    "itomo_unet_pool_fwd": ([_vp, _i, _i, _i, _i, _vp, _vp, _vp], _i),
    "itomo_unet_pool_bwd": ([_vp, _vp, _vp, _vp, _i, _i, _i, _i, _vp, _vp], _i),
    "itomo_unet_upcat_fwd": ([_vp, _vp, _i, _i, _i, _i, _i, _vp, _vp], _i),
    "itomo_unet_upcat_bwd": ([_vp, _vp, _i, _i, _i, _i, _i, _vp, _vp, _vp], _i),
    "itomo_unet_head_fwd": ([_vp, _vp, _vp, _vp, _i64, _i, _vp, _vp], _i),
    "itomo_unet_head_bwd": ([_vp, _vp, _vp, _i64, _i, _vp, _vp, _vp, _vp], _i),
    "itomo_unet_mse": ([_vp, _vp, _i64, _vp, _vp, _vp, _vp], _i),
    "itomo_unet_adam": ([_vp, _vp, _vp, _vp, _vp, _i64, _f, _f, _f, _f, _i, _vp], _i),
    "itomo_unet_to_bf16": ([_vp, _i64, _vp, _vp], _i),
    "itomo_sps_weights": ([_vp, _vp, _i, _vp, _vp, _vp, _vp, _vp], _i),
    "itomo_sps_iterate": ([_vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _vp], _i),
    "itomo_grad": ([_vp, _i, _i, _vp, _vp], _i),
    "itomo_grad_adjoint": ([_vp, _i, _i, _vp, _vp], _i),
    "itomo_cg_hp": ([_vp, _vp, _vp, _i, _i, _f, _f, _vp, _vp, _vp], _i),
    "itomo_cg_update": ([_vp, _vp, _vp, _vp, _i64, _i, _vp, _vp, _vp], _i),
    "itomo_cg_direction": ([_vp, _vp, _i64, _i, _i, _vp, _vp], _i),
    "itomo_cg_dot": ([_vp, _vp, _i64, _i, _i, _vp, _vp, _vp], _i),
    "itomo_tv_residual": ([_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _f, _vp, _vp, _vp], _i),
    "itomo_tv_rhs": ([_vp, _vp, _vp, _i64, _f, _vp], _i),
    "itomo_admm_tv_update": ([_vp, _vp, _vp, _i, _i, _f, _f, _vp, _vp, _vp], _i),
    "itomo_batch_create": ([ctypes.POINTER(_vp), _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp], _i),
    "itomo_batch_sirt_iterate": ([_vp, _f, _vp], _i),
    "itomo_batch_destroy": ([_vp], _i),
    "itomo_graph_sirt": ([ctypes.POINTER(_vp), _vp, _vp, _vp, _vp, _vp, _vp, _i, _f, _vp, _i, _vp], _i),
    "itomo_graph_batch_sirt": ([ctypes.POINTER(_vp), _vp, _f, _i, _vp], _i),
    "itomo_graph_launch": ([_vp, _vp], _i),
    "itomo_graph_destroy": ([_vp], _i),
    "itomo_filter_taps": ([_i, _i, _vp], _i),
    "itomo_gridrec_create": ([ctypes.POINTER(_vp), _i, _i, _i, _vp, _vp, _i, _i, _vp, _f, _f, _i,
                              _i, _vp, _vp, _vp], _i),
    "itomo_gridrec_destroy": ([_vp], _i),
    "itomo_gridrec_back": ([_vp, _vp, _vp, _i, _i, _vp], _i),
    "itomo_gridrec_forward": ([_vp, _vp, _vp, _i, _vp], _i),
    "itomo_fft_rows": ([_vp, _i, _i, _i, _vp], _i),
    "itomo_filter_rows": ([_vp, _vp, _i, _i, _vp, _vp], _i),
}

UNET_MSE_WORK = 1024  # ITOMO_UNET_MSE_WORK
FWD_VARIANTS = 3      # ITOMO_FWD_VARIANTS
BACK_VARIANTS = 4     # ITOMO_BACK_VARIANTS
BACK_AUTO = 255       # ITOMO_BACK_AUTO
FILTERS = {"ramp": 0, "shepp-logan": 1, "cosine": 2, "hamming": 3, "hanning": 4, "none": 5}

VEC_WORK_PER_SLICE = 771
NOALLOC_SCRATCH_BYTES = 64 << 20   # ITOMO_NOALLOC_SCRATCH_BYTES

EXPORTS = tuple(_SIGS)


def lib():
    """The loaded library (raises ItomoError when it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ItomoError(
                "libitomo.so is not built (expected at %s); run "
                "`python -m iterative_tomographic_reconstruction_algorithms_amd.build`"
                % LIB_PATH)
        L = ctypes.CDLL(LIB_PATH)
        for name, (args, res) in _SIGS.items():
            f = getattr(L, name)
            f.argtypes = args
            f.restype = res
        _lib = L
    return _lib


def check(rc, what=""):
    if rc != ITOMO_OK:
        msg = lib().itomo_last_error().decode(errors="replace")
        raise ItomoError("%s failed (status %d): %s" % (what or "itomo call", rc, msg))
    return rc
