"""ctypes binding of libezl.so (the C ABI declared in include/ezl.h).

There is no fallback: if the library is missing, or a call fails, a RuntimeError is raised.
"""
import ctypes
import functools
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "lib", "libezl.so")

_vp, _i64, _i32, _f32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float
_i64p = ctypes.POINTER(ctypes.c_int64)
_vpp = ctypes.POINTER(ctypes.c_void_p)



class Layer(ctypes.Structure):
    """struct ezl_layer"""
    _fields_ = ([(n, _i64) for n in ("s", "b", "h", "nq", "nk", "d", "f", "ndocs", "npos")] + [(n, _f32) for n in ("eps1", "eps2", "scale")]
                + [(n, _vp) for n in ("ln1", "wq", "wk", "wv", "bq", "bk", "bv", "wo", "ln2", "wg", "wu", "wd", "cos", "sin", "position_ids",
                                      "cu_seqlens")])


class LayerGrad(ctypes.Structure):
    """struct ezl_layer_grad"""
    _fields_ = [("f32", _vp), ("bf16", _vp), ("accumulate", _i32)]


_layerp = ctypes.POINTER(Layer)

# name -> argtypes; the single source of truth for the symbol table on the Python side
SIGNATURES = {
    "ezl_rmsnorm_fwd": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _f32, _vp],
    "ezl_rmsnorm_bwd": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i32, _vp, _i64, _i64, _i64, _vp],
    "ezl_rmsnorm_bwd_noalloc": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i32, _i64, _i64, _vp],
    "ezl_rmsnorm_fwd_swapped": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _f32, _vp],
    "ezl_rmsnorm_bwd_swapped": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i32, _vp, _i64, _i64, _i64, _i64, _vp],
    "ezl_swiglu_fwd": [_vp, _vp, _vp, _i64, _vp],
    "ezl_swiglu_bwd": [_vp, _vp, _vp, _vp, _vp, _i64, _vp],
    "ezl_rope_table": [_vp, _vp, _vp, _i64, _i64, _f32, _vp],
    "ezl_rope_apply": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i32, _vp],
    "ezl_rope_apply_pair": [_vp, _vp, _i64, _i64, _i64, _vp, _vp, _i64, _i64, _i64, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i32, _vp],
    "ezl_ids_in_range": [_vp, _i64, _i64, _vp, _vp],
    "ezl_ids_in_range_host_flag": [_vp, _i64, _i64, _vp, _vp],
    "ezl_embed_gather": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "ezl_embed_gather_host_flag": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "ezl_embed_scatter_add": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i32, _vp],
    "ezl_embed_grad_bf16": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "ezl_embed_gather_swapped": [_vp, _vp, _vp, _vp, _i32, _i64, _i64, _i64, _i64, _vp],
    "ezl_embed_grad_swapped": [_vp, _vp, _vp, _i32, _vp, _i64, _i64, _i64, _i64, _i64, _i32, _vp],
    "ezl_transpose01": [_vp, _vp, _i64, _i64, _i64, _vp],
    "ezl_copy_list": [_i32, _vpp, _vpp, _i64p, _vp],
    "ezl_add": [_vp, _vp, _vp, _i64, _vp],
    "ezl_cast_bf16_to_f32": [_vp, _vp, _i64, _vp],
    "ezl_cast_f32_to_bf16": [_vp, _vp, _i64, _vp],
    "ezl_bias_add": [_vp, _vp, _vp, _i64, _i64, _vp],
    "ezl_bias_grad": [_vp, _vp, _vp, _i32, _vp, _i64, _i64, _i64, _vp],
    "ezl_gemm_bf16": [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _vp, _i64, _vp],
    "ezl_gemm_bf16_ksplit": [_i32, _vpp, _vpp, _vp, _i64, _i64, _i64p, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _vp, _i64, _vp],
    "ezl_gemm_bf16_group": [_i32, _vpp, _vpp, _vpp, _i64p, _i64p, _i64, _i64p, _i64p, _i64p, _i32, _i32, _i32, ctypes.POINTER(_i32), _vp,
                            _i64, _vp],
    "ezl_attn_fwd": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _i64p, _vp],
    "ezl_attn_bwd": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _f32,
                     _i64p, _vp, _i64, _vp],
    "ezl_mask_compact": [_vp, _i64, _i64, _vp, _vp, _vp, _vp],
    "ezl_rows_gather": [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _vp],
    "ezl_ce_prepare": [_vp, _vp, _i32, _i64, _vp, _vp, _i64, _vp],
    "ezl_ce_fwd": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i32, _vp],
    "ezl_ce_bwd": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i32, _vp],
    "ezl_ce_loss": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i32, _vp],
    "ezl_ce_fused": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i32, _vp],
    "ezl_ce_reduce": [_vp, _vp, _vp, _vp, _i64, _vp],
    "ezl_scale_by_scalar": [_vp, _vp, _i64, _i32, _vp],
    "ezl_sumsq_f32": [_vp, _i64, _vp, _vp],
    "ezl_clip_coef": [_vp, _i64, _f32, _vp, _vp],
    "ezl_build_location_idx": [_vp, _i64, _vp, _i64, _i64, _i64, _i64, _vp, _i64],
    "ezl_layer_fwd": [_layerp, _vp, _vp, _vp, _vp, _vp],
    "ezl_layer_bwd": [_layerp, _vp, _vp, _vp, _vp, _vp, ctypes.POINTER(LayerGrad), _vp],
    "ezl_sumsq_list": [_i32, _vpp, _i64p, _vp, _vp],
    "ezl_adamw_list": [_i32, _vpp, _vpp, _vpp, _vpp, _vpp, _i64p, _f32, _f32, _f32, _f32, _f32, _i64, _i32, _vp, _vp],
    "ezl_adamw_step": [_vp, _vp, _vp, _vp, _vp, _i64, _f32, _f32, _f32, _f32, _f32, _i64, _i32, _vp, _vp],
}
_SPECIAL = {
    "ezl_version": ([], ctypes.c_int),
    "ezl_last_error": ([], ctypes.c_char_p),
    "ezl_rmsnorm_bwd_workspace_bytes": ([_i64, _i64], _i64),
    "ezl_rmsnorm_bwd_noalloc_max_h": ([], _i64),
    "ezl_bias_grad_workspace_bytes": ([_i64, _i64], _i64),
    "ezl_embed_scatter_add_workspace_bytes": ([_i64, _i64], _i64),
    "ezl_attn_bwd_workspace_bytes": ([_i64, _i64, _i64, _i64, _i64], _i64),
    "ezl_attn_plan": ([_i32, _i32, _i64, _i64, _i64, _i64, _i64, _i64], _i32),
    "ezl_gemm_workspace_bytes": ([_i64, _i64, _i64], _i64),
    "ezl_gemm_group_workspace_bytes": ([_i32, _i64p, _i64p, _i64], _i64),
    "ezl_gemm_group_form_workspace_bytes": ([_i32, _i32, _i64p, _i64p, _i64], _i64),
    "ezl_gemm_searches": ([], _i64),
    "ezl_gemm_plan": ([_i32, _i32, _i64p, _i64p, _i64] + [ctypes.POINTER(_i32)] * 4, _i32),
    "ezl_layer_plan": ([_layerp, _i32], _i32),
    "ezl_layer_bytes": ([_layerp, _i32], _i64),
    "ezl_sumsq_partials": ([], _i64),
    "ezl_sumsq_list_partials": ([_i32], _i64),
    "ezl_location_idx_rows": ([_i64, _i64, _i64], _i64),
}

_lib = None
_functions = {}


def exported_symbols():
    return sorted(list(SIGNATURES) + list(_SPECIAL))


def load():
    """Loads the shared library once; raises if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                "libezl.so not found at %s -- build it with `python -m easyllm_amd.csrc.build` "
                "(there is no fallback path)" % LIB_PATH)
        lib = ctypes.CDLL(LIB_PATH)
        for name, argtypes in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.argtypes = argtypes
            fn.restype = ctypes.c_int
            _functions[name] = fn
        for name, (argtypes, restype) in _SPECIAL.items():
            fn = getattr(lib, name)
            fn.argtypes = argtypes
            fn.restype = restype
        _lib = lib
    return _lib


def call(name, *args):
    """Calls an int-returning entry point and raises RuntimeError with the library's message on failure."""
    if _lib is None:
        load()
    rc = _functions[name](*args)
    if rc != 0:
        msg = _lib.ezl_last_error()
        raise RuntimeError("%s failed (%d): %s" % (name, rc, msg.decode() if msg else "?"))


def rmsnorm_bwd_workspace_bytes(rows, h):
    return load().ezl_rmsnorm_bwd_workspace_bytes(rows, h)


def bias_grad_workspace_bytes(rows, n):
    return load().ezl_bias_grad_workspace_bytes(rows, n)


def embed_scatter_add_workspace_bytes(rows, vocab):
    return load().ezl_embed_scatter_add_workspace_bytes(rows, vocab)


def attn_bwd_workspace_bytes(total_tokens, ndocs, nq, nk, d):
    return load().ezl_attn_bwd_workspace_bytes(total_tokens, ndocs, nq, nk, d)


def attn_plan(backward, ndocs, total_tokens, s_len, nq, nk, d):
    """ndocs: None without cu_seqlens"""
    documents = 0 if ndocs is None else 1
    return load().ezl_attn_plan(1 if backward else 0, documents, ndocs if documents else total_tokens // s_len, total_tokens, s_len, nq, nk, d)


@functools.lru_cache(maxsize=1024)  # a function of the sizes alone
def gemm_workspace_bytes(M, N, K):
    return load().ezl_gemm_workspace_bytes(M, N, K)


@functools.lru_cache(maxsize=1024)
def gemm_group_workspace_bytes(Ms, Ns, K):
    n = len(Ms)
    return load().ezl_gemm_group_workspace_bytes(n, (_i64 * n)(*Ms), (_i64 * n)(*Ns), K)


@functools.lru_cache(maxsize=1024)
def gemm_group_form_workspace_bytes(a_kc, Ms, Ns, K):
    n = len(Ms)
    return load().ezl_gemm_group_form_workspace_bytes(1 if a_kc else 0, n, (_i64 * n)(*Ms), (_i64 * n)(*Ns), K)


GEMM_FORMS = {"forward": 0, "weight gradient": 1, "input gradient": 2, "input gradient over pairs": 3}


def gemm_plan(form, Ms, Ns, K):
    """(one launch?, tile rows, tile columns, split, waves) of products of contiguous operands"""
    n, out = len(Ms), [_i32() for _ in range(4)]
    one = load().ezl_gemm_plan(GEMM_FORMS[form], n, (_i64 * n)(*Ms), (_i64 * n)(*Ns), K, *(ctypes.byref(x) for x in out))
    if one < 0:
        raise ValueError("gemm_plan: bad sizes")
    return (one == 1,) + tuple(x.value for x in out)


def layer_plan(layer, fp32):
    """whether a layer's weight gradients go out as one list of tiles"""
    return load().ezl_layer_plan(ctypes.byref(layer), 1 if fp32 else 0) == 1


def layer_bytes(layer, which):
    return load().ezl_layer_bytes(ctypes.byref(layer), which)


def sumsq_partials():
    return load().ezl_sumsq_partials()


def sumsq_list_partials(count):
    return load().ezl_sumsq_list_partials(count)


def location_idx_rows(seq_length, num_epochs, tokens_per_epoch):
    return load().ezl_location_idx_rows(seq_length, num_epochs, tokens_per_epoch)
