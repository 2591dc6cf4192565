"""ctypes binding of libkerops_hip.so (the C ABI declared in include/kerops_hip.h).

There is no fallback: if the library has not been built, or a call returns an
error code, a RuntimeError is raised.  `python -m kerops_amd.build` builds it.
"""
import ctypes
import importlib.machinery
import importlib.util
import os
import sys
import types
import weakref

import torch

from .settings import hardware_conf, stream_table

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, '_C', 'libkerops_hip.so')
HOST_PATH = os.path.join(_HERE, '_C', 'kerops_host.so')

KEROPS_OK = 0
KEROPS_E_BADARG = -1
KEROPS_E_UNSUPPORTED_C = -2
KEROPS_E_WORKSPACE = -3
KEROPS_E_LAUNCH = -4

# KEROPS_HIP_VERSION of include/kerops_hip.h that SIGNATURES below mirrors
HEADER_VERSION = 211

DTYPE_TAGS = {torch.float16: 0, torch.float32: 1, torch.bfloat16: 2}
# result types the gradient reduction kernels write themselves (the *_f16_out entry points)
GW_DTYPES = {torch.float16: 0, torch.float32: 1}

_p = ctypes.c_void_p
_i32 = ctypes.c_int32
_i64 = ctypes.c_int64
_f32 = ctypes.c_float

# name -> (restype, argtypes); mirrors include/kerops_hip.h one to one
SIGNATURES = {
    'kerops_hip_version': (ctypes.c_int, []),
    'kerops_last_error_string': (ctypes.c_char_p, []),
    'kerops_dwconv_fwd_f16': (ctypes.c_int, [_p, _p, _p, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _p]),
    'kerops_dwconv_stats_workspace_bytes': (_i64, [_i32, _i32, _i32, _i32, _i32]),
    'kerops_dwconv_stats_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _i64, _i32, _i32, _i32, _i32, _i32, _p]),
    'kerops_dwconv_bwd_workspace_bytes': (_i64, [_i32, _i32, _i32, _i32, _i32, _i32]),
    'kerops_dwconv_bwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _p]),
    'kerops_dwconv_bwd_f16_out': (ctypes.c_int, [_p, _p, _p, _p, _p, _i32, _p, _i64, _i32, _i32, _i32, _i32, _i32, _i32,
                                                 _p]),
    'kerops_dwconv_wgrad_workspace_bytes': (_i64, [_i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32]),
    'kerops_dwconv_wgrad_f16': (ctypes.c_int, [_p, _p, _p, _p, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
                                               _i32, _p]),
    'kerops_dwconv_wgrad_f16_out': (ctypes.c_int, [_p, _p, _p, _i32, _p, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
                                                   _i32, _i32, _p]),
    'kerops_dwconv_wgrad_noalloc_f16': (ctypes.c_int, [_p, _p, _p, _i32, _i32, _i32, _i32, _i32, _p]),
    'kerops_stats_workspace_bytes': (_i64, [_i64, _i32, _i32]),
    'kerops_stats_f16': (ctypes.c_int, [_p, _p, _p, _i64, _i32, _p, _i64, _i32, _i32, _i32, _p]),
    'kerops_stats_bwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _i64, _i32, _i32, _i32, _i32, _p]),
    'kerops_add_stats_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _i64, _i32, _p, _i64, _i32, _i32, _i32, _p]),
    'kerops_add_stats_bwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _i64, _i32, _i32, _i32, _i32, _p]),
    'kerops_bnrelu_fwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _i64, _i32, _i32, _i32, _i32, _p]),
    'kerops_bnrelu_bwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _p, _i64, _i32, _p, _i64, _i32, _i32, _i32,
                                             _p]),
    'kerops_avgpool_ceil_stats_workspace_bytes': (_i64, [_i32, _i32, _i32, _i32, _i32, _i32]),
    'kerops_avgpool_ceil_stats_f16': (ctypes.c_int, [_p, _p, _p, _p, _i32, _i32, _i32, _i32, _i32, _p, _i64, _i32,
                                                     _i32, _i32, _p]),
    'kerops_bnrelu_avgpool_ceil_stats_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _i32, _i32, _i32, _i32, _i32, _p,
                                                            _i64, _i32, _i32, _i32, _p]),
    'kerops_avgpool_ceil_stats_bwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
                                                         _i32, _p]),
    'kerops_quant_u8_window': (ctypes.c_int, [_p, _i32, _p, _i64, _f32, _i32, _i32, _i32, _p]),
    'kerops_dequant_u8_window': (ctypes.c_int, [_p, _p, _i32, _i64, _f32, _i32, _i32, _i32, _p]),
    'kerops_absmax_workspace_bytes': (_i64, [_i32]),
    'kerops_absmax_f16': (ctypes.c_int, [_p, _p, _i64, _p, _i64, _i32, _p]),
    'kerops_quant_i8_sym_f16': (ctypes.c_int, [_p, _p, _p, _p, _i64, _i32, _i32, _i32, _p]),
    'kerops_pointwise_f16': (ctypes.c_int, [_p, _p, _p, _p, _i64, _i32, _i32, _i32, _p]),
    'kerops_bnrelu_pointwise_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _i64, _i32, _i32, _p]),
    'kerops_lin_brelu_lin_add_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _i64, _i32, _p]),
    'kerops_lin_brelu_lin_bwd_workspace_bytes': (_i64, [_i64, _i32]),
    'kerops_lin_brelu_lin_bwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i32, _p]),
    'kerops_lin_brelu_lin_bwd_f16_out': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _p, _p, _p, _i32, _p, _i64, _i64, _i32,
                                                        _p]),
    'kerops_relu_linear_bwd_workspace_bytes': (_i64, [_i64, _i32, _i32]),
    'kerops_relu_linear_bwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _i64, _i64, _i32, _i32, _p]),
    'kerops_relu_linear_bwd_f16_out': (ctypes.c_int, [_p, _p, _p, _p, _p, _i32, _p, _i64, _i64, _i32, _i32, _p]),
    'kerops_bnrelu_linear_bwd_workspace_bytes': (_i64, [_i64, _i32, _i32]),
    'kerops_bnrelu_linear_bwd_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _p, _i32, _p, _p, _i64, _i64, _i32, _i32, _p]),
    'kerops_dwsep_block_workspace_bytes': (_i64, [_i32, _i32, _i32, _i32, _i32, _i32]),
    'kerops_dwsep_block_f16': (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _p, _i32, _i32, _i32, _i32, _i32, _i32, _p,
                                              _i64, _p]),
}

_lib = None
# The native call path of the ops (csrc/host.cpp), there once the library is loaded
host = None
# op name -> (ConfiguredFunction, or None for a plain function; [(dictionary, or None for its configurators, key, value),
# ...]: what has to be as it was at import for the native path to take a call)
native_ops = {}


class KeropsHipError(RuntimeError):
    def __init__(self, name, code, text):
        super().__init__(f'{name} failed with code {code}: {text}')
        self.code = code


def load():
    """Load the library once; raise if it is missing (no CPU or eager fallback exists)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f'{LIB_PATH} is missing: build the HIP extension first (python -m kerops_amd.build); '
                'kerops_amd has no fallback path'
            )
        lib = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        built = lib.kerops_hip_version()
        if built != HEADER_VERSION:
            raise RuntimeError(
                f'{LIB_PATH} reports interface version {built}, this binding was written for {HEADER_VERSION}: '
                'rebuild the library (python -m kerops_amd.build)'
            )
        _load_host(lib)
        _lib = lib
    return _lib


def _load_host(lib):
    global host
    from .ops import addition, avgpool, bnrelu, conv, fused, linear, quantization, stats  # noqa: F401 (fill native_ops)
    from .ops.conv import dwconv, dwconv_wgrad

    if not os.path.exists(HOST_PATH):
        raise RuntimeError(f'{HOST_PATH} is missing: build the HIP extension first (python -m kerops_amd.build)')
    loader = importlib.machinery.ExtensionFileLoader('kerops_host', HOST_PATH)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location('kerops_host', HOST_PATH, loader=loader))
    try:
        loader.exec_module(module)
    except ImportError as e:
        raise RuntimeError(f'{HOST_PATH} does not load ({e}): rebuild the library (python -m kerops_amd.build)') from e
    # the extension reads objects of torch and of the interpreter by the layouts of the headers it was compiled with
    built = (module.HEADER_VERSION, module.TORCH_VERSION, module.PYTHON_VERSION)
    here = (HEADER_VERSION, str(torch.__version__), sys.hexversion >> 16)
    if built != here:
        raise RuntimeError(f'{HOST_PATH} was built for (interface, torch, Python) {built}, this is {here}: '
                           'rebuild the library (python -m kerops_amd.build)')
    module.setup(
        {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in SIGNATURES},
        {name: (None if op is None else op.__dict__, [(globals(), '_lib', lib)] + entries)
         for name, (op, entries) in native_ops.items()},
        sys.modules[__name__], stream_table.__dict__, hardware_conf.__dict__, dwconv.__dict__,
        dwconv_wgrad.__dict__)
    for name, (op, _) in native_ops.items():
        if op is not None:
            op.native, op.native_for = getattr(module, name), weakref.ref(op)
    host = module


# names that csrc/host.cpp reads on every call instead of relying on what they were at import
_LIVE = frozenset(('_lib', 'host', '_table', 'SMALL_BYTES', 'L1_CACHE_BYTES', '_WAVES', '_TILE_D', '_TILE_W', '_LANE_C', 'FWD_VARIANTS',
                   'WGRAD_VARIANTS'))


def _codes(code):
    yield code
    for const in code.co_consts:
        if isinstance(const, types.CodeType):
            yield from _codes(const)


def _relied(function, found):
    """Adds to `found` ({(id of a dictionary, key): (dictionary, key, value)}) every module-level name that `function` and the
    functions of this package that it goes through read, and the attributes that they read of modules."""
    def note(owner):
        for name in names & owner.keys() - _LIVE:
            if (id(owner), name) in found:
                continue
            value = owner[name]
            found[id(owner), name] = (owner, name, value)
            if name != 'load':
                follow(value)

    def follow(value):
        if isinstance(value, types.ModuleType):
            note(vars(value))
        elif isinstance(value, types.FunctionType) and value.__module__.startswith(__package__):
            _relied(value, found)

    names = {name for code in _codes(function.__code__) for name in code.co_names} - {function.__name__}
    note(function.__globals__)
    # (modules that another function has been found to read, of which this one reads other attributes)
    for name in names & function.__globals__.keys():
        if isinstance(function.__globals__[name], types.ModuleType):
            note(vars(function.__globals__[name]))
    for cell in function.__closure__ or ():
        follow(cell.cell_contents)


def native(op):
    """Decorator of an op that csrc/host.cpp can take."""
    origin = getattr(op, 'origin_function', op)
    found = {}
    _relied(origin, found)
    entries = []
    if origin is not op:
        entries = [(op.__dict__, 'origin_function', origin)] + [(None, name, conf) for name, conf in op.configurators.items()]
        for conf in op.configurators.values():
            if isinstance(conf, types.FunctionType):
                _relied(conf, found)
    native_ops[origin.__name__] = (None if origin is op else op, list(found.values()) + entries)
    return op


def last_error():
    return load().kerops_last_error_string().decode('utf-8', 'replace')


def fail(name, code):
    raise KeropsHipError(name, code, last_error())


def call(name, *args):
    """Call an int-returning entry point and turn error codes into exceptions."""
    rc = getattr(load(), name)(*args)
    if rc != KEROPS_OK:
        fail(name, rc)
    return rc


def query(name, *args):
    """Call a *_workspace_bytes function (negative result = error)."""
    n = getattr(load(), name)(*args)
    if n < 0:
        fail(name, int(n))
    return int(n)


def ptr(t):
    return t.data_ptr() if t is not None else None


_raw_stream = getattr(torch._C, '_cuda_getCurrentRawStream', None)


def stream_of(t):
    """Raw hipStream_t of torch's current stream on the tensor's device."""
    if _raw_stream is not None:  # one C call instead of building a torch.cuda.Stream object (4 us)
        index = t.device.index
        return _raw_stream(index if index is not None else torch.cuda.current_device())
    return torch.cuda.current_stream(t.device).cuda_stream


def workspace(nbytes, device):
    """Scratch buffer owned by the caller side of the ABI (torch's caching allocator)."""
    return torch.empty(max(int(nbytes), 16), dtype=torch.uint8, device=device)

