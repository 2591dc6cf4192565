"""The measured workloads of kerops_amd: what a 3D network built on channels-last fp16 volumes asks of it.

Volumes are (N, C, H, W, D) fp16 channels_last_3d tensors.  Eight kinds of calls are covered:

  conv        DWConv: inference, and the forward half of training
  conv_grad   DWConvWGRAD (weight gradient alone: the first layer, a frozen trunk) or DWConvBackward (both gradients)
  norm_pool   Stats -> batch-norm fold -> ApplyBNReLU -> AvgPoolCeilStats, forward (a down-sampling stage)
  join        residual join and down-sampling, one training step through the plain functions: AddStats -> fold ->
              ApplyBNReLU -> AvgPoolCeilStats, then the three backward functions in reverse
  block       depthwise residual block, one training step through torch.autograd: DWConvStatsFn -> fold ->
              ApplyBNReLULinearAddFn and all gradients
  linear      ReLULinearAdd and ReLULinearBackward: pointwise channel mixing, one training step
  bottleneck  LinBReLULinAdd and LinBReLULinBackward: inverted bottleneck, one training step
  int8        DWSepBlockInt8: fused depthwise-separable inference block with int8 output
  quant       QuantUint8Window and DequantUint8Window: activations kept as bytes between two passes

Sizes run from the deepest levels of such a network (a few hundred thousand elements, where launches and host time
count) over ordinary training patches to the whole volume (1, 64, 350, 350, 128); extents need not be even.
"""
import itertools
import math

import torch

from kerops_amd.autograd import ApplyBNReLULinearAddFn, DWConvStatsFn
from kerops_amd.ops.addition import AddStats, AddStatsBackward
from kerops_amd.ops.avgpool import AvgPoolCeilStats, AvgPoolCeilStatsBackward
from kerops_amd.ops.bnrelu import ApplyBNReLU, ApplyBNReLUBackward
from kerops_amd.ops.conv import DWConv, DWConvBackward, DWConvWGRAD
from kerops_amd.ops.fused import DWSepBlockInt8
from kerops_amd.ops.linear import LinBReLULinAdd, LinBReLULinBackward, ReLULinearAdd, ReLULinearBackward
from kerops_amd.ops.quantization import DequantUint8Window, QuantUint8Window
from kerops_amd.ops.stats import Stats

DEVICE = 'cuda'
EPS = 1e-5
WINDOW = 3.0  # of the byte quantiser: activations are about N(0, 1)
DTYPES = {'fp16': torch.float16, 'bf16': torch.bfloat16, 'fp32': torch.float32}


def _case(kind, n, c, h, w, d, **more):
    return dict(kind=kind, n=n, c=c, h=h, w=w, d=d, **more)


def listed():
    cases = {
        # one sample of a small patch at the narrowest width: inference latency, one launch
        'conv_small': _case('conv', 1, 8, 64, 64, 32),
        # an ordinary training batch at an inner level
        'conv_patch': _case('conv', 2, 32, 96, 96, 96),
        # a whole volume in one piece
        'conv_volume': _case('conv', 1, 64, 350, 350, 128),
        # weight gradient of a whole volume
        'wgrad_volume': _case('conv_grad', 1, 64, 350, 350, 128, want='w'),
        # both gradients at a deep, wide level with odd extents
        'conv_grad_wide_odd': _case('conv_grad', 2, 128, 45, 51, 37, want='xw'),
        # normalise and down-sample a whole volume
        'norm_pool_volume': _case('norm_pool', 1, 64, 350, 350, 128),
        # residual join and down-sampling of a small training batch with odd extents: many short launches
        'join_odd': _case('join', 2, 16, 64, 57, 41),
        # one residual block of a patch-based training run, forward and backward
        'block_patch': _case('block', 1, 16, 128, 128, 128),
        # channel mixing behind a depthwise convolution, widening
        'linear_widen': _case('linear', 1, 64, 96, 96, 96, cout=128),
        # inverted bottleneck of a large patch
        'bottleneck_patch': _case('bottleneck', 1, 32, 175, 175, 64),
        # quantised inference block
        'int8_block': _case('int8', 1, 64, 128, 128, 128, cout=128),
        # activations of an odd-sized level stored as bytes and read back
        'quant_odd': _case('quant', 1, 16, 175, 175, 67, dtype='bf16'),
    }
    return [dict(name=name, **case) for name, case in cases.items()]


# kind -> (smallest and largest element count of the volume, channel counts)
_RANGES = {
    'conv': (1 << 18, 1003520000, (8, 16, 32, 64, 128)),
    'conv_grad': (1 << 18, 600000000, (8, 16, 32, 64, 128)),
    'norm_pool': (1 << 18, 900000000, (8, 16, 32, 64, 128)),
    'join': (1 << 18, 100000000, (8, 16, 32, 64, 128)),
    'block': (1 << 20, 100000000, (16, 32, 64, 128)),
    'linear': (1 << 18, 150000000, (16, 32, 64, 128)),
    'bottleneck': (1 << 18, 150000000, (16, 32, 64)),
    'int8': (1 << 18, 134217728, (64,)),
    'quant': (1 << 18, 440000000, (8, 16, 32, 64, 128)),
}


def draw(rng):
    kind = rng.choice(sorted(_RANGES))
    low, high, channels = _RANGES[kind]
    c = rng.choice(channels)
    elements = math.exp(rng.uniform(math.log(low), math.log(high)))
    voxels = elements / c
    n = rng.choice((1, 1, 2, 4)) if voxels >= 4096 else 1
    edge = (voxels / n) ** (1 / 3)
    h = max(4, round(edge * math.exp(rng.uniform(-0.5, 0.5))))
    d = max(4, min(256, round(edge * math.exp(rng.uniform(-0.5, 0.5)))))
    w = max(4, min(round(voxels / (n * h * d)), int(high // (n * c * h * d))))
    more = {}
    if kind == 'conv_grad':
        more['want'] = rng.choice(('w', 'xw', 'xw'))
    elif kind == 'linear':
        more['cout'] = rng.choice([o for o in (16, 32, 64, 128) if o <= 2 * c])
    elif kind == 'int8':
        more['cout'] = rng.choice((64, 128))
    elif kind == 'quant':
        more['dtype'] = rng.choice(sorted(DTYPES))
    return _case(kind, n, c, h, w, d, **more)


class _Source:
    """Inputs drawn on the GPU from one seed."""

    def __init__(self, case, seed):
        self.case = case
        self.gen = torch.Generator(DEVICE).manual_seed(seed)

    def volume(self, c=None, shape=None, mean=0.0, std=1.0, dtype=torch.float16):
        k = self.case
        n, h, w, d = shape or (k['n'], k['h'], k['w'], k['d'])
        t = torch.randn(n, h, w, d, c or k['c'], device=DEVICE, dtype=dtype, generator=self.gen)
        if (mean, std) != (0.0, 1.0):
            t.mul_(std).add_(mean)
        return t.permute(0, 4, 1, 2, 3)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(*shape, device=DEVICE, generator=self.gen) * std).to(dtype)

    def gain(self, c):
        return torch.rand(c, device=DEVICE, generator=self.gen) + 0.5

    def taps(self, c):
        return self.normal(3, 3, 3, c, std=1 / math.sqrt(27), dtype=torch.float16)

    def matrix(self, cin, cout):
        return self.normal(cin, cout, std=1 / math.sqrt(cin), dtype=torch.float16)


def prepare(case, seed):
    src = _Source(case, seed)
    kind, c = case['kind'], case['c']
    s = {'case': case}
    if kind == 'conv':
        s.update(x=src.volume(), taps=src.taps(c))
    elif kind == 'conv_grad':
        s.update(x=src.volume(), grad=src.volume())
        if case['want'] == 'xw':
            s['taps'] = src.taps(c)
    elif kind == 'norm_pool':
        s.update(x=src.volume(mean=0.5, std=math.sqrt(2.0)), gamma=src.gain(c), beta=src.normal(c, std=0.1))
    elif kind == 'join':
        pooled = (case['n'], *(-(-case[e] // 2) for e in 'hwd'))
        s.update(x=src.volume(mean=0.25), y=src.volume(mean=0.25), gamma=src.gain(c), beta=src.normal(c, std=0.1),
                 grad=src.volume(shape=pooled), grad_mean=src.normal(c), grad_sqmean=src.normal(c))
    elif kind == 'block':
        s.update(x=src.volume(mean=0.5).requires_grad_(True), taps=src.taps(c).requires_grad_(True),
                 gamma=src.gain(c).requires_grad_(True), beta=src.normal(c, std=0.1).requires_grad_(True),
                 mix=src.matrix(c, c).requires_grad_(True), grad=src.volume())
    elif kind == 'linear':
        s.update(x=src.volume(), mix=src.matrix(c, case['cout']), skip=src.volume(case['cout']),
                 grad=src.volume(case['cout']))
    elif kind == 'bottleneck':
        s.update(x=src.volume(), up=src.matrix(c, 2 * c), down=src.matrix(2 * c, c),
                 bias=src.normal(2 * c, std=0.3, dtype=torch.float16), skip=src.volume(), grad=src.volume())
    elif kind == 'int8':
        s.update(x=src.volume(), taps=src.taps(c), scale=src.gain(c), shift=src.normal(c, std=0.1),
                 mix=src.matrix(c, case['cout']))
    elif kind == 'quant':
        s.update(x=src.volume(dtype=DTYPES[case['dtype']]))
    return s


def _fold(mean, sqmean, gamma, beta):
    """Batch statistics and affine parameters -> 1/sqrt(var + eps) and the scale and shift of ApplyBNReLU."""
    rstd = torch.rsqrt(sqmean - mean * mean + EPS)
    scale = gamma * rstd
    return rstd, scale, beta - mean * scale


def _norm_pool(s):
    mean, sqmean = Stats(s['x'])
    _, scale, shift = _fold(mean, sqmean, s['gamma'], s['beta'])
    act = ApplyBNReLU(s['x'], scale, shift)
    pooled, pmean, psqmean = AvgPoolCeilStats(act)
    return {'mean': mean, 'sqmean': sqmean, 'act': act, 'pooled': pooled, 'pmean': pmean, 'psqmean': psqmean}


def _join(s):
    z, mean, sqmean = AddStats(s['x'], s['y'])
    rstd, scale, shift = _fold(mean, sqmean, s['gamma'], s['beta'])
    act = ApplyBNReLU(z, scale, shift)
    pooled, pmean, psqmean = AvgPoolCeilStats(act)
    dact = AvgPoolCeilStatsBackward(s['grad'], s['grad_mean'], s['grad_sqmean'], pooled, tuple(act.shape))
    dz, dscale, dshift = ApplyBNReLUBackward(z, scale, shift, dact)
    # back through the fold
    centred = dscale - mean * dshift
    dgamma = centred * rstd
    dvar = -0.5 * rstd * rstd * scale * centred
    dmean = -scale * dshift - 2.0 * mean * dvar
    dx = AddStatsBackward(dz, dmean, dvar, z)
    return {'z': z, 'mean': mean, 'sqmean': sqmean, 'pooled': pooled, 'pmean': pmean, 'psqmean': psqmean, 'dx': dx,
            'dgamma': dgamma, 'dbeta': dshift}


def _block(s):
    y, mean, sqmean = DWConvStatsFn.apply(s['x'], s['taps'])
    _, scale, shift = _fold(mean, sqmean, s['gamma'], s['beta'])
    out = ApplyBNReLULinearAddFn.apply(y, scale, shift, s['mix'], s['x'])
    names = ('x', 'taps', 'gamma', 'beta', 'mix')
    grads = torch.autograd.grad(out, [s[k] for k in names], s['grad'])
    return {'out': out.detach(), **{'d' + k: g for k, g in zip(names, grads)}}


def run(state):
    s = state
    kind = s['case']['kind']
    if kind == 'conv':
        return DWConv(s['x'], s['taps'])
    if kind == 'conv_grad':
        if s['case']['want'] == 'w':
            return DWConvWGRAD(s['x'], s['grad'])
        return DWConvBackward(s['x'], s['grad'], s['taps'])
    if kind == 'norm_pool':
        return _norm_pool(s)
    if kind == 'join':
        return _join(s)
    if kind == 'block':
        return _block(s)
    if kind == 'linear':
        out = ReLULinearAdd(s['x'], s['mix'], s['skip'])
        dx, dmix = ReLULinearBackward(s['x'], s['grad'], s['mix'])
        return {'out': out, 'dx': dx, 'dmix': dmix}
    if kind == 'bottleneck':
        out = LinBReLULinAdd(s['x'], s['up'], s['down'], s['bias'], s['skip'])
        dx, dup, ddown, dbias = LinBReLULinBackward(s['x'], s['grad'], s['up'], s['down'], s['bias'])
        return {'out': out, 'dx': dx, 'dup': dup, 'ddown': ddown, 'dbias': dbias}
    if kind == 'int8':
        q, qscale, y = DWSepBlockInt8(s['x'], s['taps'], s['scale'], s['shift'], s['mix'])
        return {'q': q, 'qscale': qscale, 'y': y}
    if kind == 'quant':
        q = QuantUint8Window(s['x'], WINDOW)
        return {'q': q, 'back': DequantUint8Window(q, s['x'].dtype, WINDOW)}
    raise ValueError(kind)


def work(case):
    """Every input read once and every output written once; multiply and add count as two."""
    kind, c = case['kind'], case['c']
    v = case['n'] * case['h'] * case['w'] * case['d']
    e = v * c
    pe = case['n'] * c * math.prod(-(-case[k] // 2) for k in 'hwd')
    if kind == 'conv':
        return {'bytes': 4 * e, 'flops': 54 * e}
    if kind == 'conv_grad':
        return {'bytes': 4 * e, 'flops': 54 * e} if case['want'] == 'w' else {'bytes': 6 * e, 'flops': 108 * e}
    if kind == 'norm_pool':
        return {'bytes': 4 * e + 2 * pe, 'flops': 10 * e}
    if kind == 'join':  # x, y, pooled gradient in; z, pooled, dx out
        return {'bytes': 8 * e + 4 * pe, 'flops': 30 * e}
    if kind == 'block':  # x and the gradient in; out and dx out
        return {'bytes': 8 * e, 'flops': (3 * 54 + 3 * 2 * c + 30) * e}
    if kind == 'linear':  # x, skip, gradient in; out, dx out
        o = v * case['cout']
        return {'bytes': 4 * e + 6 * o, 'flops': 6 * v * c * case['cout']}
    if kind == 'bottleneck':  # x, skip, gradient in; out, dx out
        return {'bytes': 10 * e, 'flops': (4 + 10) * 2 * c * e}
    if kind == 'int8':  # x in; y and its int8 form out
        o = v * case['cout']
        return {'bytes': 2 * e + 3 * o, 'flops': 54 * e + 2 * v * c * case['cout']}
    size = DTYPES[case['dtype']].itemsize
    return {'bytes': (2 * size + 1) * e, 'flops': 8 * e}


# Four times the difference of each kind from the same formulas in 64 bits at (2,16,24,23,21), (1,64,21,22,20) and
# (2,32,40,41,39), as measured (rel, max):
#   conv, conv_grad  one rounding to fp16: 2.2e-4, 4.9e-4
#   norm_pool        two roundings: 2.4e-4, 8.7e-4
#   linear           product and sum rounded to fp16: 2.5e-4, 1.2e-3
#   int8             y 3.0e-4, 1.6e-3; 0.5 % of the int8 values fall on the other side of a rounding boundary
#   join, block, bottleneck
#                    outputs 3.1e-4; gradients up to 9e-3, where a rounding moves a value across the ReLU's zero, and
#                    there a single element of an input gradient differs by its full size
_TOLERANCE = {
    'conv': {'rel': 1e-3, 'max': 2e-3},
    'conv_grad': {'rel': 1e-3, 'max': 2e-3},
    'norm_pool': {'rel': 1e-3, 'max': 4e-3},
    'linear': {'rel': 1e-3, 'max': 5e-3},
    'int8': {'rel': 1.2e-3, 'max': 6e-3, 'differ': 0.01},
    'join': {'rel': 3e-2, 'max': 0.99},
    'block': {'rel': 3e-2, 'max': 0.99},
    'bottleneck': {'rel': 3e-2, 'max': 0.99},
    'quant': 'exact',
}


def tolerance(case):
    return _TOLERANCE[case['kind']]


def _conv64(x, taps):
    """Depthwise 3x3x3 convolution with zero padding of an (N, H, W, D, C) tensor."""
    _, h, w, d, _ = x.shape
    padded = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    y = torch.zeros_like(x)
    for i, j, k in itertools.product(range(3), repeat=3):
        y = y + padded[:, i:i + h, j:j + w, k:k + d] * taps[i, j, k]
    return y


def _taps_grad64(x, grad):
    _, h, w, d, c = x.shape
    padded = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = torch.empty(3, 3, 3, c, device=x.device, dtype=x.dtype)
    for i, j, k in itertools.product(range(3), repeat=3):
        out[i, j, k] = (padded[:, i:i + h, j:j + w, k:k + d] * grad).sum((0, 1, 2, 3))
    return out


def _pool64(x):
    """2x2x2 ceil-mode average over the voxels that exist, and the statistics of the result."""
    def halved(t):
        t = torch.nn.functional.pad(t, (0, 0, *(e for n in reversed(t.shape[1:4]) for e in (0, n % 2))))
        n, h, w, d, c = t.shape
        return t.view(n, h // 2, 2, w // 2, 2, d // 2, 2, c).sum((2, 4, 6))

    pooled = halved(x) / halved(torch.ones_like(x[:1, ..., :1]))
    return pooled, *_stats64(pooled)


def _stats64(x):
    return x.mean((0, 1, 2, 3)), (x * x).mean((0, 1, 2, 3))


def exact(case, seed):
    """The outputs of `run` in plain torch and 64 bits.  Bytes are no computed numbers: None stands in their place."""
    kind = case['kind']
    s = {}
    for key, t in prepare(case, seed).items():
        if torch.is_tensor(t):
            t = t.detach().double()
            s[key] = t.permute(0, 2, 3, 4, 1) if t.ndim == 5 else t

    def volume(t):
        return t.detach().permute(0, 4, 1, 2, 3)

    def grads(outputs, upstream, names):
        got = torch.autograd.grad(outputs, [s[k] for k in names], upstream)
        return {k: volume(g) if g.ndim == 5 else g for k, g in zip(names, got)}

    def differentiable(*names):
        for k in names:
            s[k] = s[k].requires_grad_(True)

    if kind == 'conv':
        return volume(_conv64(s['x'], s['taps']))
    if kind == 'conv_grad':
        dtaps = _taps_grad64(s['x'], s['grad'])
        if case['want'] == 'w':
            return dtaps
        return volume(_conv64(s['grad'], s['taps'].flip(0, 1, 2))), dtaps
    if kind == 'norm_pool':
        mean, sqmean = _stats64(s['x'])
        _, scale, shift = _fold(mean, sqmean, s['gamma'], s['beta'])
        act = torch.relu(s['x'] * scale + shift)
        pooled, pmean, psqmean = _pool64(act)
        return {'mean': mean, 'sqmean': sqmean, 'act': volume(act), 'pooled': volume(pooled), 'pmean': pmean,
                'psqmean': psqmean}
    if kind == 'join':
        s['z'] = s['x'] + s['y']
        differentiable('z', 'gamma', 'beta')
        mean, sqmean = _stats64(s['z'])
        _, scale, shift = _fold(mean, sqmean, s['gamma'], s['beta'])
        pooled, pmean, psqmean = _pool64(torch.relu(s['z'] * scale + shift))
        g = grads((pooled, pmean, psqmean), (s['grad'], s['grad_mean'], s['grad_sqmean']), ('z', 'gamma', 'beta'))
        return {'z': volume(s['z']), 'mean': mean.detach(), 'sqmean': sqmean.detach(), 'pooled': volume(pooled),
                'pmean': pmean.detach(), 'psqmean': psqmean.detach(), 'dx': g['z'], 'dgamma': g['gamma'],
                'dbeta': g['beta']}
    if kind == 'block':
        names = ('x', 'taps', 'gamma', 'beta', 'mix')
        differentiable(*names)
        y = _conv64(s['x'], s['taps'])
        _, scale, shift = _fold(*_stats64(y), s['gamma'], s['beta'])
        out = torch.relu(y * scale + shift) @ s['mix'] + s['x']
        return {'out': volume(out), **{'d' + k: g for k, g in grads(out, s['grad'], names).items()}}
    if kind == 'linear':
        differentiable('x', 'mix')
        out = torch.relu(s['x']) @ s['mix'] + s['skip']
        return {'out': volume(out), **{'d' + k: g for k, g in grads(out, s['grad'], ('x', 'mix')).items()}}
    if kind == 'bottleneck':
        names = ('x', 'up', 'down', 'bias')
        differentiable(*names)
        out = torch.relu(s['x'] @ s['up'] + s['bias']) @ s['down'] + s['skip']
        return {'out': volume(out), **{'d' + k: g for k, g in grads(out, s['grad'], names).items()}}
    if kind == 'int8':
        y = torch.relu(_conv64(s['x'], s['taps']) * s['scale'] + s['shift']) @ s['mix']
        return {'q': None, 'qscale': y.abs().amax() / 127, 'y': volume(y)}
    if kind == 'quant':
        level = ((s['x'].clamp(-WINDOW, WINDOW) + WINDOW) / (2 * WINDOW) * 255).floor()
        return {'q': None, 'back': volume(level * (2 * WINDOW / 255) - WINDOW)}
    raise ValueError(kind)
