"""CPU tests of the C-ABI boundary: the built library loads, exports every symbol the header
declares, validates arguments before touching a device, and the Python ops keep the
reference's host-side contract checks (same exception types, raised before the ABI is
crossed).  No kernel is launched here."""
import ctypes
import os
import re

import pytest
import torch

from kerops_amd import _lib
from kerops_amd.settings import CongiguratorError

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, 'include', 'kerops_hip.h')


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r'/\*.*?\*/', '', text, flags=re.S)
    return sorted(set(re.findall(r'\b(kerops_[a-z0-9_]+)\s*\(', text)))


def header_version():
    return int(re.search(r'#define\s+KEROPS_HIP_VERSION\s+(\d+)', open(HEADER).read()).group(1))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    names = declared_symbols()
    assert len(names) >= 20
    for name in names:
        assert hasattr(lib, name), f'{name} is declared in include/kerops_hip.h but not exported'
    # and the ctypes table binds exactly the declared set
    assert sorted(_lib.SIGNATURES) == names
    assert lib.kerops_hip_version() == _lib.HEADER_VERSION == header_version()


def test_argument_validation_needs_no_device():
    lib = _lib.load()
    rc = lib.kerops_dwconv_fwd_f16(None, None, None, 1, 4, 4, 4, 8, 0, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_BADARG and 'pointer' in _lib.last_error()
    buf = (ctypes.c_char * 4096)()
    addr = (ctypes.addressof(buf) + 15) & ~15
    rc = lib.kerops_dwconv_fwd_f16(addr, addr, addr, 1, 4, 4, 4, 24, 0, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_UNSUPPORTED_C
    rc = lib.kerops_dwconv_fwd_f16(addr, addr, addr, 1, 4, 4, 4, 64, 5, 7, 0, 2, None)
    assert rc == _lib.KEROPS_E_BADARG and 'no kernel built' in _lib.last_error()
    rc = lib.kerops_dwconv_fwd_f16(addr + 2, addr, addr, 1, 4, 4, 4, 64, 0, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_BADARG
    rc = lib.kerops_dwconv_wgrad_f16(addr, addr, addr, addr, 16, 1, 4, 4, 4, 64, 0, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_WORKSPACE
    # the typed-result variants take fp32 or fp16 only, and check it before anything else
    rc = lib.kerops_dwconv_wgrad_f16_out(addr, addr, addr, 2, addr, 1 << 30, 1, 4, 4, 4, 64, 0, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_BADARG and 'gw_dtype' in _lib.last_error()
    rc = lib.kerops_dwconv_bwd_f16_out(addr, addr, addr, addr, addr, 7, addr, 1 << 30, 1, 4, 4, 4, 64, 0, None)
    assert rc == _lib.KEROPS_E_BADARG and 'gw_dtype' in _lib.last_error()
    rc = lib.kerops_dwconv_wgrad_f16_out(addr, addr, addr, 0, addr, 16, 1, 4, 4, 4, 64, 0, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_WORKSPACE
    rc = lib.kerops_relu_linear_bwd_f16_out(addr, addr, addr, addr, addr, 2, addr, 1 << 30, 64, 32, 32, None)
    assert rc == _lib.KEROPS_E_BADARG and 'dw_dtype' in _lib.last_error()
    rc = lib.kerops_lin_brelu_lin_bwd_f16_out(addr, addr, addr, addr, addr, addr, addr, addr, addr, -1, addr, 1 << 30,
                                              64, 32, None)
    assert rc == _lib.KEROPS_E_BADARG and 'grad_dtype' in _lib.last_error()
    rc = lib.kerops_stats_f16(addr, addr, addr, 64, 1024, addr, 1 << 30, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_UNSUPPORTED_C
    rc = lib.kerops_stats_f16(addr, addr, addr, 64, 12, addr, 1 << 30, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_BADARG
    rc = lib.kerops_quant_u8_window(addr, 7, addr, 16, 1.0, 0, 0, 0, None)
    assert rc == _lib.KEROPS_E_BADARG and 'dtype' in _lib.last_error()
    # launch-shape knobs of the stream kernels: wavefronts per workgroup in {4, 8, 16}, segment in {1, 4, 8}
    for waves, segment, word in [(5, 0, 'waves'), (32, 1, 'waves'), (4, 2, 'segment'), (16, 16, 'segment')]:
        rc = lib.kerops_bnrelu_fwd_f16(addr, addr, addr, addr, 64, 64, 0, waves, segment, None)
        assert rc == _lib.KEROPS_E_BADARG and word in _lib.last_error()
    rc = lib.kerops_stats_f16(addr, addr, addr, 64, 64, addr, 1 << 30, 70000, 0, 0, None)
    assert rc == _lib.KEROPS_E_BADARG and 'blocks' in _lib.last_error()


def test_every_entry_point_rejects_null_pointers_before_touching_the_device():
    # all pointers null, all sizes a plausible 16 / 1.0: every compute entry point must come back with an error
    # code and a message (no launch, no dereference), so that a caller's mistake never reaches the GPU
    lib = _lib.load()
    for name, (res, argtypes) in _lib.SIGNATURES.items():
        if res is not ctypes.c_int or not any(a is ctypes.c_void_p for a in argtypes):
            continue
        args = [None if a is ctypes.c_void_p else (1.0 if a is ctypes.c_float else 16) for a in argtypes]
        rc = getattr(lib, name)(*args)
        assert rc in (_lib.KEROPS_E_BADARG, _lib.KEROPS_E_UNSUPPORTED_C, _lib.KEROPS_E_WORKSPACE), (name, rc)
        assert _lib.last_error(), name


def test_extreme_sizes_never_reach_a_launch():
    # sizes up to INT32_MAX with null pointers, and every workspace query over a grid of extreme extents: the
    # host arithmetic (grid planning, workspace sizes) must neither crash nor report success for a null pointer
    import itertools
    lib = _lib.load()
    for name, (res, argtypes) in _lib.SIGNATURES.items():
        if 'workspace_bytes' in name:
            for vals in itertools.product([1, 8, 64, 350, 2 ** 31 - 1], repeat=min(len(argtypes), 5)):
                n = getattr(lib, name)(*(list(vals) + [0] * (len(argtypes) - len(vals))))
                assert n >= _lib.KEROPS_E_LAUNCH, (name, vals, n)  # a size or one of the error codes
        elif res is ctypes.c_int and any(a is ctypes.c_void_p for a in argtypes):
            for v in (0, 1, 7, 65535, 2 ** 31 - 1):
                args = [None if a is ctypes.c_void_p else (1.0 if a is ctypes.c_float else v) for a in argtypes]
                assert getattr(lib, name)(*args) < 0, (name, v)


def test_workspace_queries():
    lib = _lib.load()
    assert lib.kerops_stats_workspace_bytes(1000, 64, 16) == 16 * 2 * 64 * 4
    assert lib.kerops_stats_workspace_bytes(1000, 64, 0) == 4096 * 2 * 64 * 4  # covers every built-in shape
    assert lib.kerops_stats_workspace_bytes(1000, 24, 16) == _lib.KEROPS_E_BADARG
    n = lib.kerops_dwconv_wgrad_workspace_bytes(1, 350, 350, 128, 64, 0, 0, 0, 0)
    assert n > 0 and n % (27 * 64 * 4) == 0  # one [27][64] fp32 partial per workgroup
    assert lib.kerops_dwconv_wgrad_workspace_bytes(1, 8, 8, 8, 24, 0, 0, 0, 0) == _lib.KEROPS_E_UNSUPPORTED_C
    assert lib.kerops_avgpool_ceil_stats_workspace_bytes(1, 7, 7, 7, 8, 4) == 4 * 2 * 8 * 4
    assert lib.kerops_absmax_workspace_bytes(10) == 40


def test_wgrad_launch_knobs_are_checked_before_any_division():
    # a zero or negative patch extent beside non-zero knobs used to divide by zero on the host
    lib = _lib.load()
    buf = (ctypes.c_char * 4096)()
    addr = (ctypes.addressof(buf) + 15) & ~15
    for tw, td, cl in [(0, 8, 16), (8, 0, 16), (0, 8, 0), (-8, 8, 16), (8, -8, 16), (8, 8, -16), (8, 8, 0),
                       (2 ** 31 - 1, 8, 16)]:
        assert lib.kerops_dwconv_wgrad_workspace_bytes(1, 16, 16, 16, 64, tw, td, 0, cl) == _lib.KEROPS_E_BADARG
        assert 'no kernel built' in _lib.last_error()
        rc = lib.kerops_dwconv_wgrad_f16(addr, addr, addr, addr, 1 << 40, 1, 16, 16, 16, 64, tw, td, 0, cl, None)
        assert rc == _lib.KEROPS_E_BADARG
    # the fused block checks plane and volume limits like the other convolution entry points
    assert lib.kerops_dwsep_block_workspace_bytes(1, 4, 2 ** 20, 2 ** 20, 64, 128) == _lib.KEROPS_E_BADARG
    assert lib.kerops_dwsep_block_workspace_bytes(2 ** 31 - 1, 2 ** 31 - 1, 256, 256, 64, 128) == _lib.KEROPS_E_BADARG


def test_split_of_the_h_march():
    # workgroup counts of the built-in launch shapes, read back from the workspace sizes (one partial per
    # workgroup).  The matrix-core convolution kernels use the balanced split by default: never more workgroups than
    # the GPU holds at once (512 of 512 threads, 1024 of 256), all of them busy at the large shapes.  Uniform chunks
    # on request: patches x chunks.
    lib = _lib.load()

    def wgrad_blocks(n, h, w, d, c, h_chunk=0):
        return lib.kerops_dwconv_wgrad_workspace_bytes(n, h, w, d, c, 0, 0, h_chunk, 0) // (27 * min(c, 64) * 4)

    def bwd_blocks(n, h, w, d, c, h_chunk=0):
        return lib.kerops_dwconv_bwd_workspace_bytes(n, h, w, d, c, h_chunk) // (27 * min(c, 64) * 4)

    def stats_blocks(n, h, w, d, c):
        return lib.kerops_dwconv_stats_workspace_bytes(n, h, w, d, c) // (2 * min(c, 64) * 4)

    for blocks in (wgrad_blocks, bwd_blocks, stats_blocks):
        assert blocks(1, 350, 350, 128, 64) == 512   # 8 groups of 64 (weight gradient: 4 rows of 16 patches)
        assert blocks(1, 350, 350, 128, 128) == 512  # the same patches in 2 slabs
        assert blocks(1, 128, 128, 128, 64) == 512
    assert wgrad_blocks(1, 350, 350, 128, 8) in range(480, 513)  # 512-thread workgroups at every channel count
    assert wgrad_blocks(1, 1, 8, 8, 8) == 1 and stats_blocks(1, 1, 8, 8, 64) == 1 and bwd_blocks(1, 1, 8, 8, 64) == 1
    assert wgrad_blocks(1, 350, 350, 128, 64, 175) == 1408 and bwd_blocks(1, 350, 350, 128, 64, 175) == 1408  # 8x8 patches
    assert wgrad_blocks(1, 350, 350, 128, 64, -32) == 512 and bwd_blocks(1, 350, 350, 128, 64, -32) == 512
    # a group that is not a multiple of the two slabs of 128 channels is refused
    assert lib.kerops_dwconv_wgrad_workspace_bytes(1, 350, 350, 128, 128, 0, 0, -3, 0) == _lib.KEROPS_E_BADARG
    assert lib.kerops_dwconv_bwd_workspace_bytes(1, 350, 350, 128, 128, -3) == _lib.KEROPS_E_BADARG


def cl3d(*shape, dtype=torch.float16):
    return torch.zeros(*shape, dtype=dtype).to(memory_format=torch.channels_last_3d)


def test_ops_keep_reference_contract_checks():
    from kerops_amd.ops.avgpool import AvgPoolCeilStats
    from kerops_amd.ops.bnrelu import ApplyBNReLU, ApplyBNReLUBackward
    from kerops_amd.ops.conv import DWConv, DWConvWGRAD
    from kerops_amd.ops.stats import Stats

    x = cl3d(1, 8, 4, 4, 4)
    w = torch.zeros(3, 3, 3, 8, dtype=torch.float16)
    with pytest.raises(AssertionError):  # not channels_last_3d
        DWConv(torch.zeros(1, 8, 4, 4, 4, dtype=torch.float16), w)
    with pytest.raises(AssertionError):  # dtype
        DWConv(x.float(), w.float())
    with pytest.raises(AssertionError):  # weight layout
        DWConv(x, torch.zeros(8, 1, 3, 3, 3, dtype=torch.float16))
    with pytest.raises(CongiguratorError):  # channel count with no launch table entry
        DWConv(cl3d(1, 4, 4, 4, 4), torch.zeros(3, 3, 3, 4, dtype=torch.float16))
    with pytest.raises(CongiguratorError):
        DWConvWGRAD(cl3d(1, 256, 2, 2, 2), cl3d(1, 256, 2, 2, 2))
    with pytest.raises(KeyError):
        DWConv(x, w, ACCTYPE='bfloat16')
    with pytest.raises(AssertionError):
        DWConvWGRAD(x, cl3d(1, 8, 4, 4, 5))
    with pytest.raises(AssertionError):  # non power of two
        Stats(cl3d(1, 6, 4, 4, 4))
    with pytest.raises(AssertionError):
        ApplyBNReLU(x, torch.zeros(4), torch.zeros(8))
    with pytest.raises(AssertionError):  # fp32 weight / bias required by the backward
        ApplyBNReLUBackward(x, torch.zeros(8, dtype=torch.float64), torch.zeros(8, dtype=torch.float64), x)
    with pytest.raises(AssertionError):  # D*C above the reference's row limit
        AvgPoolCeilStats(cl3d(1, 128, 2, 2, 512))


def test_no_cpu_fallback():
    from kerops_amd.ops.conv import DWConv
    from kerops_amd.ops.quantization import QuantUint8Window
    from kerops_amd.ops.stats import Stats

    x = cl3d(1, 8, 4, 4, 4)
    with pytest.raises(RuntimeError, match='no CPU path'):
        DWConv(x, torch.zeros(3, 3, 3, 8, dtype=torch.float16))
    with pytest.raises(RuntimeError, match='no CPU path'):
        Stats(x)
    with pytest.raises(RuntimeError, match='no CPU path'):
        QuantUint8Window(x, 1.0)


def test_missing_library_fails_loudly(monkeypatch):
    monkeypatch.setattr(_lib, '_lib', None)
    monkeypatch.setattr(_lib, 'LIB_PATH', os.path.join(ROOT, 'kerops_amd', '_C', 'does_not_exist.so'))
    with pytest.raises(RuntimeError, match='no fallback'):
        _lib.load()


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, 'kerops_amd')
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith(('.py', '.hip', '.hpp', '.h', '.cpp')):
                text = open(os.path.join(dirpath, f)).read()
                assert 'import oracle' not in text and 'from oracle' not in text and 'oracle/' not in text, f


def test_built_in_split_never_exceeds_the_resident_workgroups():
    # chunks of H are only taken where they run in one round: the partial sums of the built-in weight-gradient shapes
    # fit the 4 MB that the entry point without a workspace owns, at any size
    import random
    lib = _lib.load()
    rng = random.Random(3)
    for _ in range(3000):
        c = rng.choice((8, 16, 32, 64, 128))
        n, h, w, d = rng.choice((1, 2, 4)), rng.randint(1, 400), rng.randint(1, 400), rng.randint(1, 256)
        partial = 27 * min(c, 64) * 4
        for need in (lib.kerops_dwconv_wgrad_workspace_bytes(n, h, w, d, c, 0, 0, 0, 0),
                     lib.kerops_dwconv_bwd_workspace_bytes(n, h, w, d, c, 0)):
            assert 0 < need <= 512 * partial < 4 << 20, (n, c, h, w, d, need // partial)
        assert lib.kerops_dwconv_stats_workspace_bytes(n, h, w, d, c) <= 1024 * 2 * min(c, 64) * 4


def test_linear_backward_takes_a_third_workgroup_in_large_volumes():
    # rows of partial sums = workgroups: two per compute unit of 256, three where half a million voxels and more keep them
    # busy (32 -> 32 lost 5 % at 15.7 M voxels with two, 16 -> 128 lost 6 % at 4 M)
    lib = _lib.load()
    for cin, cout in ((32, 32), (16, 128)):
        small, large = (lib.kerops_relu_linear_bwd_workspace_bytes(v, cin, cout) for v in (200000, 4000000))
        assert large * 2 == small * 3, (cin, cout, small, large)
    # the widest pair holds two workgroups in LDS
    assert (lib.kerops_relu_linear_bwd_workspace_bytes(4000000, 128, 128)
            == lib.kerops_relu_linear_bwd_workspace_bytes(200000, 128, 128) == 512 * 128 * 128 * 4)


def test_built_in_split_gives_two_rows_where_workgroups_share_a_compute_unit():
    # a workgroup that marches over one row of H reads three planes for it: only where each has a compute unit of its own
    # (the fused backward, which keeps one row per workgroup up to all slots, is the faster for it)
    lib = _lib.load()

    def partials(name, n, c, h, w, d, rows):
        wgrad = name == 'kerops_dwconv_wgrad_workspace_bytes'
        return getattr(lib, name)(n, h, w, d, c, *((0, 0, rows, 0) if wgrad else (rows,))) // (27 * min(c, 64) * 4)

    wgrad, fused = 'kerops_dwconv_wgrad_workspace_bytes', 'kerops_dwconv_bwd_workspace_bytes'
    for shape in ((2, 32, 32, 9, 35), (2, 128, 10, 36, 11), (1, 16, 30, 57, 33), (1, 16, 26, 44, 43), (1, 32, 44, 32, 28)):
        assert partials(wgrad, *shape, 1) > 256
        assert 0 < partials(wgrad, *shape, 0) <= partials(wgrad, *shape, 2), shape
        assert partials(fused, *shape, 0) == partials(fused, *shape, 1) <= 512, shape
    for shape in ((1, 32, 33, 19, 25), (1, 64, 21, 11, 30), (4, 32, 12, 13, 15), (1, 32, 1, 64, 64)):
        assert partials(wgrad, *shape, 0) == partials(wgrad, *shape, 1) <= 256, shape


def test_bnrelu_linear_backward_entry_point_refuses():
    lib = _lib.load()
    buf = (ctypes.c_char * 4096)()
    at = (ctypes.addressof(buf) + 15) & ~15
    need = lib.kerops_bnrelu_linear_bwd_workspace_bytes(100, 16, 32)
    assert need == 1 * (16 * 32 + 2 * 16) * 4  # one workgroup: its weight gradient, its scale and shift sums

    def call(x=at, scale=at, shift=at, g=at, wm=at, dx=at, dw=at, dtype=0, daffine=at, ws=at, nbytes=need, v=100, cin=16,
             cout=32):
        return lib.kerops_bnrelu_linear_bwd_f16(x, scale, shift, g, wm, dx, dw, dtype, daffine, ws, nbytes, v, cin, cout, None)

    for bad in (dict(x=None), dict(scale=None), dict(shift=None), dict(g=None), dict(wm=None), dict(dx=None), dict(dw=None),
                dict(daffine=None), dict(x=at + 8), dict(g=at + 2), dict(wm=at + 8), dict(dx=at + 8), dict(dtype=2),
                dict(dtype=7), dict(v=0), dict(v=-5)):
        assert call(**bad) == _lib.KEROPS_E_BADARG, bad
        assert 'bnrelu_linear_bwd' in _lib.last_error()
    for bad in (dict(ws=None), dict(ws=at + 4), dict(nbytes=need - 1), dict(nbytes=0), dict(nbytes=-1)):
        assert call(**bad) == _lib.KEROPS_E_WORKSPACE, bad
    for cin, cout in ((8, 16), (16, 8), (24, 16), (256, 16), (16, 0), (-16, 16)):
        assert call(cin=cin, cout=cout) == _lib.KEROPS_E_UNSUPPORTED_C
        assert lib.kerops_bnrelu_linear_bwd_workspace_bytes(100, cin, cout) == _lib.KEROPS_E_UNSUPPORTED_C
    assert lib.kerops_bnrelu_linear_bwd_workspace_bytes(0, 16, 16) == _lib.KEROPS_E_BADARG


def test_bnrelu_linear_backward_checks_its_tensors():
    from kerops_amd.ops.linear import ApplyBNReLULinearBackward

    def call(x=cl3d(1, 16, 4, 4, 4), scale=torch.zeros(16), shift=torch.zeros(16), grad=cl3d(1, 32, 4, 4, 4),
             weight=torch.zeros(16, 32, dtype=torch.float16)):
        return ApplyBNReLULinearBackward(x, scale, shift, grad, weight)

    for bad in (dict(x=cl3d(1, 16, 4, 4, 4).float()), dict(x=torch.zeros(1, 16, 4, 4, 4, dtype=torch.float16)),
                dict(grad=cl3d(1, 32, 4, 4, 5)), dict(grad=cl3d(2, 32, 4, 4, 4)), dict(scale=torch.zeros(8)),
                dict(shift=torch.zeros(32)), dict(weight=torch.zeros(32, 16, dtype=torch.float16)),
                dict(weight=torch.zeros(16, 32)), dict(grad=torch.zeros(1, 32, 4, 4, 4, dtype=torch.float16)),
                dict(x=cl3d(1, 8, 4, 4, 4), scale=torch.zeros(8), shift=torch.zeros(8),
                     weight=torch.zeros(8, 32, dtype=torch.float16))):
        with pytest.raises(AssertionError):
            call(**bad)
    with pytest.raises(RuntimeError, match='no CPU path'):
        call()
