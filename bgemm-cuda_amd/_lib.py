"""ctypes binding of libbgemm_mi355x.so (the C ABI declared in include/bgemm_mi355x.h).

The library must have been built (``python _build.py`` or ``__graft_entry__.build()``);
there is no CPU fallback: a missing library raises ImportError.
"""
import ctypes
import importlib.machinery
import importlib.util
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
SO_PATH = os.path.join(_HERE, "libbgemm_mi355x.so")
NATIVE_PATH = os.path.join(_HERE, "_bgemm_native.so")

OK, EINVAL, ENULL, EWORKSPACE, ELAUNCH, EALIGN, ETIMEOUT = 0, -1, -2, -3, -4, -5, -6
MODE_AND, MODE_XOR, MODE_ATTN, MODE_BWTA, MODE_ATTN_X = 0, 1, 2, 3, 4
OUT_I32, OUT_F16, OUT_F32_SCALED, OUT_F16_SCALED, OUT_BITS_F32, OUT_BITS_F16 = 0, 1, 2, 3, 4, 5
SRC_F16, SRC_F32, SRC_BITS = 0, 1, 2
ABI_VERSION = 12
NATIVE_VERSION = 2     # of the native part's functions (torch_common.h): another when one is added or called another way
LAYOUT_VERSION = 6     # of the tiled operand layout, written into packed files; changes only when the layout does
STATIC_SCRATCH_BYTES = 32 << 20      # BGEMM_STATIC_SCRATCH_BYTES
VARIANT_AUTO, VARIANT_VALU, VARIANT_MFMA, VARIANT_MFMA_F4 = 0, 1, 2, 3
# BGEMM_KERNEL_*: what bgemm_packed_kernel_id() returns and force_kernel() takes
KERNEL_MFMA_256x256, KERNEL_MFMA_128x128, KERNEL_MFMA_64x128, KERNEL_MFMA_32x128, KERNEL_MFMA_256x128 = 0, 1, 2, 3, 4
KERNEL_MFMA_32x256, KERNEL_MFMA_64x64, KERNEL_MFMA_128x64, KERNEL_MFMA_128x256T = 5, 6, 7, 8
KERNEL_SKINNY_STREAM, KERNEL_SKINNY_SPLITK, KERNEL_SKINNY_QUAD, KERNEL_SKINNY_POPC, KERNEL_VALU = 16, 17, 18, 19, 32


def force_kernel(kernel_id, family=VARIANT_AUTO):
    """BGEMM_FORCE_KERNEL(id) | family: a `variant` that runs the named kernel whatever the shape (tests, benchmarks)."""
    return ((kernel_id + 1) << 8) | family


_i64, _p, _int, _sz = ctypes.c_int64, ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t

# symbol -> (restype, argtypes); mirrors include/bgemm_mi355x.h one to one
SIGNATURES = {
    "bgemm_last_error": (ctypes.c_char_p, []),
    "bgemm_abi_version": (_int, []),
    "bgemm_tiled_words": (_i64, [_i64, _i64]),
    "bgemm_pack_sign_f16": (_int, [_p, _i64, _i64, _i64, _p, _p]),
    "bgemm_pack_sign_f16_logical": (_int, [_p, _i64, _i64, _i64, _p, _p]),
    "bgemm_pack_sign_centered": (_int, [_p, _int, _i64, _i64, _i64, _p, _p, _p]),
    "bgemm_pack_ternary_f16": (_int, [_p, _i64, _i64, _i64, _p, _p, _p]),
    "bgemm_tile_from_logical": (_int, [_p, _i64, _i64, _p, _p]),
    "bgemm_logical_from_tiled": (_int, [_p, _i64, _i64, _p, _p]),
    "bgemm_packed_workspace_bytes": (_sz, [_int, _i64, _i64, _i64, _i64, _int, _int]),
    "bgemm_packed_counter_bytes": (_sz, [_int, _i64, _i64, _i64, _i64, _int, _int]),
    "bgemm_packed_forward": (_int, [_int, _p, _p, _p, _p, _int, _i64, _i64, _i64, _i64, _i64, _i64, _i64,
                                    _int, _int, _p, _sz, _p, _sz, _p]),
    "bgemm_packed_kernel_id": (_int, [_int, _int, _i64, _i64, _i64, _i64, _int, _int]),
    "bgemm_row_popcounts": (_int, [_p, _i64, _i64, _i64, _i64, _p, _p]),
    "bgemm_packed_forward_counted": (_int, [_int, _p, _p, _p, _p, _p, _int, _i64, _i64, _i64, _i64, _i64, _i64, _i64,
                                            _int, _p]),
    "bgemm_packed_forward_scaled": (_int, [_int, _p, _p, _p, _p, _int, _i64, _i64, _i64, _i64, _i64, _i64, _i64,
                                           _int, _int, _p, _sz, _p, _sz, _p, _p, _p, _p]),
    "bgemm_packed_forward_bits": (_int, [_int, _p, _p, _p, _p, _int, _i64, _i64, _i64, _i64, _i64, _i64, _i64,
                                         _int, _int, _p, _sz, _p, _sz, _p, _p, _p, _p, _p]),
    "bgemm_pack_sign_f16_transposed": (_int, [_p, _i64, _i64, _i64, _i64, _i64, _p, _p]),
    "bgemm_pack_batched": (_int, [_p, _int, _int, _p, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _p, _p, _p]),
    "bgemm_pack_transposed_batched": (_int, [_p, _int, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _p, _p]),
    "bgemm_packed_weight_forward_supported": (_int, [_int, _i64, _i64, _i64]),
    "bgemm_packed_weight_forward": (_int, [_int, _p, _p, _int, _i64, _p, _p, _int, _i64, _i64, _i64, _int, _p, _p, _p, _p, _p]),
    "bgemm_unpacked_workspace_bytes": (_sz, [_int, _p, _int, _i64, _i64, _i64, _i64]),
    "bgemm_unpacked_workspace_bytes_on": (_sz, [_int, _p, _int, _i64, _i64, _i64, _i64, _p]),
    "bgemm_unpacked_forward": (_int, [_int, _p, _p, _int, _i64, _p, _p, _int, _i64, _i64, _i64, _p, _p, _p, _p, _sz, _p]),
    "bgemm_f16_workspace_bytes": (_sz, [_i64, _i64, _i64, _int]),
    "bgemm_f16_forward": (_int, [_p, _p, _p, _i64, _i64, _i64, _p, _sz, _int, _int, _p]),
    "bgemm_f16_forward_static": (_int, [_p, _p, _p, _i64, _i64, _i64, _int, _int, _p]),
    "bgemm_pack_sign_nonzero_pair": (_int, [_p, _i64, _i64, _p, _p, _p, _p, _i64, _i64, _p, _p, _p, _int, _i64, _p]),
    "bgemm_linear_backward_workspace_bytes": (_sz, [_i64, _i64, _i64, _int, _int]),
    "bgemm_linear_train_forward": (_int, [_p, _i64, _p, _p, _i64, _p, _int, _i64, _i64, _i64, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p]),
    "bgemm_linear_backward": (_int, [_p, _p, _p, _p, _p, _int, _i64, _i64, _i64, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _sz, _p]),
    "bgemm_elastic_forward": (_int, [_p, _p, _i64, _i64, _i64, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p]),
    "bgemm_elastic_backward_workspace_bytes": (_sz, [_i64, _i64, _i64, _int, _int]),
    "bgemm_elastic_backward": (_int, [_p, _p, _p, _p, _p, _p, _p, ctypes.c_float, _i64, _i64, _i64, _p, _p, _p, _p, _p, _p, _sz, _p]),
    "bgemm_linear_rows_supported": (_int, [_i64, _i64, _i64, _int, _int]),
    "bgemm_linear_rows_forward": (_int, [_p, _int, _i64, _i64, _i64, _i64, _int, _p, _int, _p, _int, _p]),
    "bgemm_linear_rows_norm_supported": (_int, [_i64, _i64, _i64]),
    "bgemm_linear_rows_norm_forward": (_int, [_p, _i64, _i64, _i64, _p, _p, _p, _p, ctypes.c_double, _p]),
    "bgemm_attention_supported": (_int, [_i64, _i64, _i64, _i64]),
    "bgemm_attention_forward": (_int, [_p, _p, _p, _i64, _i64, _i64, _i64, _p, _p, _int, _p]),
    "bgemm_attention_forward_bits": (_int, [_p, _p, _p, _i64, _i64, _i64, _i64, _p, _p, _p, _int, _p]),
    "bgemm_scores_forward": (_int, [_int, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _p, _p]),
    "bgemm_context_forward": (_int, [_p, _p, _p, _i64, _i64, _i64, _i64, _i64, _p, _p]),
    "bgemm_scores_backward": (_int, [_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _p, _p, _p]),
    "bgemm_context_backward": (_int, [_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _p, _p, _p]),
    "bgemm_chain_workspace_bytes": (_sz, [_int, _p, _int, _i64]),
    "bgemm_chain_forward": (_int, [_int, _p, _p, _int, _p, _p, _i64, _p, _int, _int, _p, _sz, _int, _p]),
    "bgemm_chain_status": (_int, [_p, _p]),
}


class RowsLayer(ctypes.Structure):
    """bgemm_rows_layer: one layer of bgemm_linear_rows_forward; every pointer is a device pointer."""
    _fields_ = [(name, _p) for name in ("W_tiled", "zero_point", "sw", "sa", "bias", "next_zero_point", "out")]


class ChainLayer(ctypes.Structure):
    """bgemm_chain_layer: one layer of a chain; every pointer is a device pointer."""
    _fields_ = [("W_tiled", _p), ("sw", _p), ("bias", _p), ("sa", _p), ("next_zero_point", _p),
                ("M", _i64), ("K", _i64), ("reserved", _i64)]

_lib = None


def lib():
    """Loads the shared library once and types every entry point."""
    global _lib
    if _lib is None:
        if not os.path.exists(SO_PATH):
            raise ImportError("%s is missing: build it with `python %s`" %
                              (SO_PATH, os.path.join(_HERE, "_build.py")))
        L = ctypes.CDLL(SO_PATH)
        version = L.bgemm_abi_version()        # before the entry points are looked up: an older library has not all of them
        if version != ABI_VERSION:
            raise ImportError("%s is ABI version %d, this binding needs %d: rebuild it" % (SO_PATH, version, ABI_VERSION))
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name, None)
            if fn is None:
                raise ImportError("%s has no %s: rebuild it" % (SO_PATH, name))
            fn.restype, fn.argtypes = res, args
        _lib = L
    return _lib


_native = None


def native():
    """The native host side of the layers (_bgemm_native.so, built with the library)."""
    global _native
    if _native is None:
        lib()                                  # the same library, with its version checked
        if not os.path.exists(NATIVE_PATH):
            raise ImportError("%s is missing: build it with `python %s`" % (NATIVE_PATH, os.path.join(_HERE, "_build.py")))
        import torch                           # noqa: F401  (its libraries must be loaded first)
        loader = importlib.machinery.ExtensionFileLoader("_bgemm_native", NATIVE_PATH)
        spec = importlib.util.spec_from_file_location("_bgemm_native", NATIVE_PATH, loader=loader)
        module = importlib.util.module_from_spec(spec)
        loader.exec_module(module)
        for name, needed in (("abi_version", ABI_VERSION), ("native_version", NATIVE_VERSION)):
            version = getattr(module, name, None)
            if version != needed:
                raise ImportError("%s states %s %s, this binding needs %d: rebuild it" % (NATIVE_PATH, name, version, needed))
        _native = module
    return _native


_native_looked_for = False


def native_or_none():
    """native() if it has been built, else None: for calls that have a form without it.  One that is there and does not load says so on
    every call."""
    global _native_looked_for
    if _native is None and not _native_looked_for:
        if os.path.exists(NATIVE_PATH):
            return native()
        _native_looked_for = True
    return _native


def native_for(dtypes, *tensors):
    """native() for a call whose tensors (or Nones) are all of one of `dtypes`, else None: what cannot be a call for it does not
    need it to be there."""
    if _native is not None:
        return _native
    first = tensors[0].dtype
    if first not in dtypes or any(t is not None and getattr(t, "dtype", None) != first for t in tensors):
        return None
    return native()


class BgemmError(RuntimeError):
    pass


def check(rc):
    """Turns a negative status into the Python exception the reference's asserts map to."""
    if rc == OK:
        return
    msg = lib().bgemm_last_error().decode() or "error %d" % rc
    if rc in (EINVAL, ENULL, EALIGN, EWORKSPACE):
        raise ValueError(msg)
    raise BgemmError(msg)
