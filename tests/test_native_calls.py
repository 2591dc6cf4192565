"""The native call path of the ops against their Python functions: the same results, shapes, strides and types wherever it
takes a call, and None for every call that it leaves to them."""
import copy
import functools
import sys

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from conftest import cpu_gen, rand_cl3d, rand_dw_weight
from kerops_amd import _lib
from kerops_amd.ops.addition import AddStats, AddStatsBackward
from kerops_amd.ops.avgpool import ApplyBNReLUAvgPoolCeilStats, AvgPoolCeilStats, AvgPoolCeilStatsBackward
from kerops_amd.ops.bnrelu import ApplyBNReLU, ApplyBNReLUBackward
from kerops_amd.ops.conv import DWConv, DWConvBackward, DWConvStats, DWConvWGRAD
from kerops_amd.ops.fused import DWSepBlock
from kerops_amd.ops.linear import (ApplyBNReLULinearAdd, ApplyBNReLULinearBackward, LinBReLULinAdd, LinBReLULinBackward,
                                   ReLULinearAdd, ReLULinearBackward)
from kerops_amd.ops.quantization import DequantUint8Window, QuantInt8Sym, QuantUint8Window
from kerops_amd.ops.stats import Stats, StatsBackward
from kerops_amd.settings import stream_table

DEV = 'cuda:0'
OPS = {op.__name__: op for op in (
    DWConv, DWConvStats, DWConvBackward, DWConvWGRAD, Stats, StatsBackward, AddStats, AddStatsBackward, ApplyBNReLU,
    ApplyBNReLUBackward, AvgPoolCeilStats, ApplyBNReLUAvgPoolCeilStats, AvgPoolCeilStatsBackward, ReLULinearAdd,
    ReLULinearBackward, ApplyBNReLULinearAdd, ApplyBNReLULinearBackward, LinBReLULinAdd, LinBReLULinBackward, QuantUint8Window,
    DequantUint8Window, QuantInt8Sym, DWSepBlock)}
GRADS = ('DWConvBackward', 'DWConvWGRAD', 'ReLULinearBackward', 'LinBReLULinBackward')  # take out_dtype
FORMS = {'plain': (2, 16, 6, 5, 4), 'odd': (1, 64, 5, 7, 3), 'flat': (1, 16, 1, 1, 33), 'single': (1, 64, 1, 1, 1), 'sliced': (1, 16, 4, 3, 5)}


def arguments(name, form, dev):
    n, c, h, w, d = FORMS[form]
    g = cpu_gen(c + h)
    big = form == 'sliced'  # one sample of a larger batch: its N stride is not that of a dense tensor

    def volume(channels=c, size=(h, w, d)):
        t = rand_cl3d(g, n + big, channels, *size).to(dev)
        return t[1:] if big else t

    def vec():
        return torch.randn(c, generator=g).to(dev)

    def matrix(cin, cout):
        return (torch.randn(cin, cout, generator=g) / cin ** 0.5).half().to(dev)

    taps = rand_dw_weight(g, c)[1].to(dev)
    half = [-(-e // 2) for e in (h, w, d)]
    return {
        'DWConv': lambda: (volume(), torch.nn.Parameter(taps)), 'DWConvStats': lambda: (volume(), taps),
        'DWConvBackward': lambda: (volume(), volume(), taps), 'DWConvWGRAD': lambda: (volume(), volume()),
        'Stats': lambda: (volume(),), 'StatsBackward': lambda: (volume(), vec(), vec()),
        'AddStats': lambda: (volume(), volume()), 'AddStatsBackward': lambda: (volume(), vec(), vec(), volume()),
        'ApplyBNReLU': lambda: (volume().requires_grad_(True), vec(), vec().reshape(1, c, 1, 1, 1)),
        'ApplyBNReLUBackward': lambda: (volume(), torch.nn.Parameter(vec().reshape(1, c)), vec(), volume()),
        'AvgPoolCeilStats': lambda: (volume(),), 'ApplyBNReLUAvgPoolCeilStats': lambda: (volume(), vec(), vec()),
        'AvgPoolCeilStatsBackward': lambda: (volume(c, half), vec(), vec(), volume(c, half), torch.Size((n, c, h, w, d))),
        'ReLULinearAdd': lambda: (volume(), matrix(c, 32), volume(32)),
        'ReLULinearBackward': lambda: (volume(), volume(32), matrix(c, 32)),
        'ApplyBNReLULinearAdd': lambda: (volume(), vec(), vec(), matrix(c, 32), volume(32)),
        'ApplyBNReLULinearBackward': lambda: (volume(), vec(), vec(), volume(32), matrix(c, 32)),
        'LinBReLULinAdd': lambda: (volume(), matrix(c, 2 * c), matrix(2 * c, c), matrix(1, 2 * c)[0], volume()),
        'LinBReLULinBackward': lambda: (volume(), volume(), matrix(c, 2 * c), matrix(2 * c, c), matrix(1, 2 * c)[0]),
        'QuantUint8Window': lambda: (volume().bfloat16(), 2.5),
        'DequantUint8Window': lambda: (volume().to(torch.uint8), torch.float32, 2.5),
        'QuantInt8Sym': lambda: (volume(), torch.full((1,), 3.0, device=dev)),
        'DWSepBlock': lambda: (volume(), taps, vec(), vec(), matrix(c, 128)),
    }[name]()


def python_function(name, args, monkeypatch, **kwargs):
    with monkeypatch.context() as m:
        m.setattr(_lib, 'host', None)
        op = OPS[name]
        if hasattr(op, 'origin_function'):
            m.setattr(op, 'native', None)
        return op(*args, **kwargs)


def same(a, b):
    a, b = [(t,) if isinstance(t, torch.Tensor) else t for t in (a, b)]
    assert type(a) is type(b) and len(a) == len(b)
    for s, t in zip(a, b):
        assert type(s) is type(t) and (s.dtype, s.device, s.shape, s.stride(), s.requires_grad) == (
            t.dtype, t.device, t.shape, t.stride(), t.requires_grad)
        assert torch.equal(s.contiguous().reshape(-1).view(torch.uint8), t.contiguous().reshape(-1).view(torch.uint8))


@pytest.fixture
def host():
    _lib.load()
    return _lib.host


def test_every_op_has_its_native_call(host):
    assert set(OPS) == set(_lib.native_ops)
    for name, op in OPS.items():
        assert callable(getattr(host, name))
        assert not hasattr(op, 'origin_function') or op.native is getattr(host, name)


@pytest.mark.parametrize('name', OPS)
def test_cpu_tensors_are_left_to_the_python_function(host, name):
    args = arguments(name, 'plain', 'cpu')
    assert getattr(host, name)(*args) is None
    with pytest.raises(RuntimeError, match='no CPU path'):
        OPS[name](*args)
    assert getattr(host, name)() is None and getattr(host, name)(*args, None) is None


def test_missing_native_calls_fail_loudly(monkeypatch):
    monkeypatch.setattr(_lib, '_lib', None)
    monkeypatch.setattr(_lib, 'HOST_PATH', _lib.HOST_PATH + '.none')
    with pytest.raises(RuntimeError, match='build the HIP extension'):
        _lib.load()


@pytest.mark.parametrize('owner,name,value', [(torch, '__version__', '2.9.1+rocm6.4'), (sys, 'hexversion', sys.hexversion + (1 << 16)),
                                              (_lib, 'HEADER_VERSION', _lib.HEADER_VERSION + 1)])
def test_native_calls_built_for_another_version_are_refused(host, monkeypatch, owner, name, value):
    lib = _lib.load()
    monkeypatch.setattr(owner, name, value)
    with pytest.raises(RuntimeError, match='rebuild the library'):
        _lib._load_host(lib)
    assert _lib.host is host


# what the Python function of an op reads of this package when it is called
READ = {'AvgPoolCeilStatsBackward': {'stream_shape', 'require_cuda', 'stream_waves', 'ceil', '_find', 'call', 'stream_of'},
        'Stats': {'numel_no_channels', 'require_cuda', 'stream_waves', 'next_power_of_2', 'query', 'workspace', '_find'},
        'QuantUint8Window': {'_dense', 'require_cuda', 'stream_waves', 'BUILT_WAVES'},
        'DWConv': {'warps', 'dblock', 'wtile', 'lanec', 'nearest_conv_shape', 'require_cuda', 'next_power_of_2', 'load'},
        'DWConvStats': {'cl3d', 'require_cuda', 'next_power_of_2', 'workspace'}}


@pytest.mark.parametrize('name', OPS)
def test_everything_that_a_python_function_reads_is_compared(host, name):
    found = {}
    _lib._relied(getattr(OPS[name], 'origin_function', OPS[name]), found)
    compared = {(id(owner), key) for owner, key, _ in _lib.native_ops[name][1]}
    assert set(found) <= compared, 'a name defined behind its op'  # (the list is made where the op is defined)
    assert READ.get(name, set()) <= {key for _, key, _ in _lib.native_ops[name][1]}
    assert not hasattr(OPS[name], 'origin_function') or (id(OPS[name].__dict__), 'origin_function') in compared


@pytest.mark.gpu
@pytest.mark.parametrize('name', OPS)
def test_a_call_with_a_replaced_name_is_left_to_the_python_function(host, monkeypatch, name):
    args = arguments(name, 'plain' if name != 'DWSepBlock' else 'odd', DEV)
    call = getattr(host, name)
    assert call(*args) is not None
    for owner, key, value in _lib.native_ops[name][1]:
        if owner is None:
            owner = OPS[name].configurators
        if owner.get('__name__', '').split('.')[0] == 'torch' or not callable(value) or isinstance(value, type):
            continue
        with monkeypatch.context() as m:
            m.setitem(owner, key, functools.partial(value))
            assert call(*args) is None, key
        assert call(*args) is not None, key


def _clone(op):
    return functools.wraps(op)(type(op)(op.origin_function, op.signature, op.configurable_args, op.usual_args, **op.configurators))


COPIES = {'copy': copy.copy, 'deepcopy': copy.deepcopy, 'wraps': _clone}


@pytest.mark.parametrize('how', COPIES)
def test_a_copy_goes_by_its_own_configurators(host, monkeypatch, how):
    taken = []
    monkeypatch.setattr(DWConvBackward, 'native', lambda *args, **kwargs: taken.append(args))
    other = COPIES[how](DWConvBackward)
    for op, native in ((DWConvBackward, True), (other, False)):
        with pytest.raises(RuntimeError, match='no CPU path'):
            op(*arguments('DWConvBackward', 'plain', 'cpu'))
        assert bool(taken) == native
        taken.clear()


@pytest.mark.gpu
@pytest.mark.parametrize('how', COPIES)
def test_a_reconfigured_copy_and_its_original(host, how):
    args = arguments('DWConvBackward', 'plain', DEV)
    other = COPIES[how](DWConvBackward)
    other.reconfigure(**{**DWConvBackward.configurators, 'out_dtype': torch.float32})
    assert other(*args)[1].dtype == torch.float32 and DWConvBackward(*args)[1].dtype == torch.float16
    assert host.DWConvBackward(*args) is not None


# (16-channel forms only where the fused block, built for 64 input channels, is not the op)
CASES = [(name, form) for name in OPS for form in FORMS if name != 'DWSepBlock' or FORMS[form][1] == 64]


@pytest.mark.gpu
@pytest.mark.parametrize('name,form', CASES)
def test_native_call_equals_the_python_function(host, monkeypatch, name, form):
    args = arguments(name, form, DEV)
    out = getattr(host, name)(*args)
    assert out is not None
    same(out, python_function(name, args, monkeypatch))
    same(OPS[name](*args), out)
    if name in GRADS:
        for dtype in (torch.float32, torch.float16):
            same(getattr(host, name)(*args, out_dtype=dtype), python_function(name, args, monkeypatch, out_dtype=dtype))
        assert getattr(host, name)(*args, out_dtype=torch.bfloat16) is None
        assert OPS[name](*args, out_dtype=torch.bfloat16)[-1].dtype == torch.bfloat16 or name == 'DWConvWGRAD'


class _Plain(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _PlainDispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
def test_unusual_calls_are_left_to_the_python_function(host, monkeypatch):
    x, taps = arguments('DWConv', 'plain', DEV)
    want = host.DWConv(x, taps)
    # modes, subclasses, copies
    for mode in (_Plain, _PlainDispatch):
        with mode():
            assert host.DWConv(x, taps) is None
            same(DWConv(x, taps), want)
    with torch.inference_mode():
        assert host.DWConv(x, taps).is_inference() and python_function('DWConv', (x, taps), monkeypatch).is_inference()
    sub = x.as_subclass(type('Sub', (torch.Tensor,), {}))
    assert host.DWConv(sub, taps) is None and torch.equal(DWConv(sub, taps).as_subclass(torch.Tensor), want)
    spread = taps.detach().transpose(0, 1).contiguous().transpose(0, 1)
    assert not spread.is_contiguous() and host.DWConv(x, spread) is None
    same(DWConv(x, spread), want)
    assert torch.vmap(lambda t: torch.tensor(host.Stats(t) is None))(x[None]).all()
    # wrong arguments: the op's own checks speak
    for bad in ((x.float(), taps), (x.contiguous(), taps), (x, taps[..., :8]), (x[0], taps)):
        assert host.DWConv(*bad) is None
        with pytest.raises((AssertionError, ValueError, IndexError)):
            DWConv(*bad)
    # the library's refusals: its own error, as from the Python function
    empty = x[:0]
    for call in (lambda: Stats(empty), lambda: python_function('Stats', (empty,), monkeypatch)):
        with pytest.raises(_lib.KeropsHipError, match='kerops_stats'):
            call()
    # a helper or a configurator replaced
    with monkeypatch.context() as m:
        called = []
        inner = _lib.call
        m.setattr(_lib, 'call', lambda *a: called.append(a[0]) or inner(*a))
        same(DWConv(x, taps), want)
        assert called == ['kerops_dwconv_fwd_f16']
    with monkeypatch.context() as m:
        m.setattr('kerops_amd.ops.conv.dwconv.dblock', lambda channels, depth=None: 16)
        assert host.DWConv(x, taps) is None
    before = dict(DWConv.configurators)
    DWConv.reconfigure(**{**before, 'H_chunk': 2})
    try:
        assert host.DWConv(x, taps) is None
        same(DWConv(x, taps), want)
    finally:
        DWConv.reconfigure(**before)
    assert host.DWConv(x, taps) is not None


@pytest.mark.gpu
def test_live_launch_tables(host, monkeypatch):
    # what the tables say at the moment of the call, as in the Python function
    (x,) = arguments('Stats', 'plain', DEV)
    with monkeypatch.context() as m:
        m.setattr(stream_table, '_table', {})
        same(host.Stats(x), python_function('Stats', (x,), monkeypatch))
        for shape in (dict(blocks=3, num_warps=8, segment=4), dict(blocks=1, num_warps=4, segment=1)):
            for key in ('small', '16', 'default'):
                m.setattr(stream_table, '_table', {})
                stream_table.set_stream_shape('Stats', key=key, **shape)
                same(host.Stats(x), python_function('Stats', (x,), monkeypatch))
        stream_table.set_stream_shape('Stats', key='default', num_warps=2)  # not built: mapped by the Python function
        assert host.Stats(x) is None
        Stats(x)


@pytest.mark.gpu
def test_native_calls_on_streams_threads_and_in_a_graph(host):
    import threading
    x, taps = arguments('DWConvStats', 'plain', DEV)
    want = DWConvStats(x, taps)
    failed = []

    def work():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(50):
                    got = host.DWConvStats(x, taps)
                torch.cuda.current_stream().synchronize()
                same(got, want)
        except BaseException as e:  # noqa: BLE001 (reported by the main thread)
            failed.append(e)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not failed, failed
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = host.DWConvStats(x, taps)
    for _ in range(3):
        [t.zero_() for t in out]
        graph.replay()
        torch.cuda.synchronize()
        same(out, want)
