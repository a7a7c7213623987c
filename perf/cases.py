"""The work that users of this framework have it do, as cases to be timed.

Two kinds of caller are represented.  One builds a Tile program (edsl / op) and runs it through `Runner` with arrays in
host memory: there a pass is the whole call, transfers included.  The other keeps tensors on the GPU and calls the
kernel library's C ABI (`hipkernels`, dispatch once / invoke many): there a pass is the invokes of one contraction or
block.  A case is a dict of plain values; `kind` names the family, the rest its sizes and options:

  network   a ResNet-50 forward pass (bf16, weights constant), input staged as the benchmark harness stages it
  dense     a stack of dense layers relu(x . W + b), weights constant, `widths` the layer widths, any of them odd
  backward  both gradients of a 2-D convolution: with respect to its data and to its filter
  batched   softmax(Q . K^T / sqrt(d)) . V over a batch of independent matrices
  rows      an operation along the rows of a matrix: mvn with scale and shift, softmax, topk or argmax
  gemm      one matrix product on the GPU with its usual tail (bias and ReLU; for int8 a requantisation to int8)
  conv      one NHWC convolution on the GPU with bias and ReLU (int8: the int32 sums)
  block     depthwise 3x3, pointwise with scale / shift / ReLU, 3x3 stride-2 max-pool with window argmax, on the GPU
"""
import ctypes
import math

import numpy as np
import torch

from plaidml_amd import edsl as P
from plaidml_amd import hipkernels as hk
from plaidml_amd import op as Pop
from plaidml_amd import resnet50

ES = {'f32': 4, 'f32x3': 4, 'bf16': 2, 'i8': 1}


def listed():
    return [
        # the smallest whole call: one example through four dense layers (the toy_gemms network), latency of a request
        {'name': 'dense_f32_b1', 'kind': 'dense', 'dtype': 'f32', 'batch': 1, 'widths': '256-512-1024-2048-1000'},
        # dense layers whose widths are no multiple of anything, a few hundred rows, bf16
        {'name': 'dense_bf16_odd', 'kind': 'dense', 'dtype': 'bf16', 'batch': 300, 'widths': '1001-777-1000'},
        # one image through a whole network: latency, many small launches
        {'name': 'resnet50_bf16_b1', 'kind': 'network', 'batch': 1},
        # the throughput configuration of the same network
        {'name': 'resnet50_bf16_b128', 'kind': 'network', 'batch': 128},
        # a training step's share of a convolution: both gradients of the 3x3 64-channel layer at a batch of 16
        {'name': 'backward_f32_3x3', 'kind': 'backward', 'dtype': 'f32', 'n': 16, 'hw': 56, 'ci': 64, 'co': 64, 'k': 3, 'stride': 1},
        # products under batch dimensions with a softmax between them
        {'name': 'batched_bf16', 'kind': 'batched', 'dtype': 'bf16', 'batch': 96, 'rows': 128, 'cols': 128, 'd': 64},
        # normalisation of rows, the element-wise and reduction path
        {'name': 'rows_mvn_f32', 'kind': 'rows', 'op': 'mvn', 'dtype': 'f32', 'rows': 4096, 'cols': 1000},
        # single fp32 product, B as it lies
        {'name': 'gemm_f32_1024', 'kind': 'gemm', 'dtype': 'f32', 'm': 1024, 'n': 1024, 'k': 1024, 'b': 'kn'},
        # the large bf16 product, both operands new in every call
        {'name': 'gemm_bf16_4096', 'kind': 'gemm', 'dtype': 'bf16', 'm': 4096, 'n': 4096, 'k': 4096, 'b': 'kn'},
        # quantised product with per-column requantisation
        {'name': 'gemm_i8_4096', 'kind': 'gemm', 'dtype': 'i8', 'm': 4096, 'n': 4096, 'k': 4096, 'b': 'kn'},
        # the benchmark's convolution, filter given with the call
        {'name': 'conv3x3_bf16_b128', 'kind': 'conv', 'dtype': 'bf16', 'n': 128, 'hw': 56, 'ci': 64, 'co': 64, 'k': 3, 'stride': 1, 'packed': False},
        # a depthwise-separable block with its pooling
        {'name': 'block_bf16_b64', 'kind': 'block', 'n': 64, 'hw': 19, 'c': 728},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['network', 'dense', 'dense', 'backward', 'backward', 'batched', 'batched', 'rows', 'rows', 'gemm', 'gemm', 'gemm',
                       'conv', 'conv', 'block'])
    if kind == 'network':
        return {'kind': kind, 'batch': _log(rng, 2, 96)}
    if kind == 'dense':
        widths = [_log(rng, 10, 2048) for _ in range(rng.randint(2, 5))]
        return {'kind': kind, 'dtype': rng.choice(['f32', 'bf16']), 'batch': _log(rng, 1, 2048), 'widths': '-'.join(map(str, widths))}
    if kind == 'backward':
        while True:
            c = {'kind': kind, 'dtype': rng.choice(['f32', 'bf16']), 'n': _log(rng, 1, 32), 'hw': _log(rng, 7, 112), 'ci': _log(rng, 3, 256),
                 'co': _log(rng, 16, 256), 'k': rng.choice([1, 3, 3, 5]), 'stride': rng.choice([1, 1, 2])}
            if _backward_flops(c) <= _backward_flops(listed()[4]):
                return c
    if kind == 'batched':
        while True:
            c = {'kind': kind, 'dtype': rng.choice(['f32', 'bf16']), 'batch': _log(rng, 1, 128), 'rows': _log(rng, 16, 512),
                 'cols': _log(rng, 16, 512), 'd': rng.choice([32, 64, 64, 80, 100, 128])}
            if c['batch'] * c['rows'] * c['cols'] <= 4 << 20:
                return c
    if kind == 'rows':
        op = rng.choice(['mvn', 'softmax', 'topk', 'argmax'])
        cols = _log(rng, 16, 2000 if op == 'topk' else 8000)
        return {'kind': kind, 'op': op, 'dtype': rng.choice(['f32', 'bf16']), 'cols': cols, 'rows': max(1, min(_log(rng, 1, 8192), (4 << 20) // cols))}
    if kind == 'gemm':
        dtype = rng.choice(['f32', 'f32x3', 'bf16', 'bf16', 'i8', 'i8'])
        k = _log(rng, 32, 4096) // 16 * 16
        return {'kind': kind, 'dtype': dtype, 'm': _log(rng, 1, 4096), 'n': _log(rng, 16, 4096), 'k': k, 'b': rng.choice(['kn', 'nk', 'packed'])}
    if kind == 'conv':
        while True:
            dtype = rng.choice(['f32', 'bf16', 'bf16', 'i8'])
            c = {'kind': kind, 'dtype': dtype, 'n': _log(rng, 1, 128), 'hw': _log(rng, 7, 150), 'ci': rng.choice([3, 16, 32, 64, 64, 96, 128, 256]),
                 'co': _log(rng, 16, 256), 'k': rng.choice([1, 3, 3, 5, 7]), 'stride': rng.choice([1, 1, 2]), 'packed': rng.choice([True, False])}
            if _conv_flops(c) <= 1.5 * _conv_flops(listed()[10]) and c['n'] * c['hw'] ** 2 * max(c['ci'], c['co']) <= 32 << 20:
                return c
    return {'kind': 'block', 'n': _log(rng, 1, 64), 'hw': _log(rng, 10, 38) if rng.random() < 0.5 else 19, 'c': 8 * _log(rng, 8, 91)}


# ---- what a pass cannot do without ---------------------------------------------------------------------

def _out(hw, stride):
    return (hw + stride - 1) // stride  # SAME


def _valid_taps(hw, k, stride):
    """Pairs (output position, tap) along one axis whose tap falls inside the image, SAME padding."""
    oh = _out(hw, stride)
    pad = max(0, (oh - 1) * stride + k - hw) // 2
    return sum(1 for y in range(oh) for t in range(k) if 0 <= y * stride + t - pad < hw)


def _conv_flops(c):
    return 2.0 * c['n'] * _valid_taps(c['hw'], c['k'], c['stride']) ** 2 * c['ci'] * c['co']


def _backward_flops(c):
    return 2.0 * _conv_flops(c)


def work(case):
    c, kind = case, case['kind']
    if kind == 'network':
        # 4.09 G multiply-adds an image at 224 x 224, 25.5 M weights in bf16, the image in bf16, 1000 results
        return {'flops': 2 * 4.09e9 * c['batch'], 'bytes': 2 * 25.5e6 + c['batch'] * (2 * 224 * 224 * 3 + 2 * 1000)}
    es = ES[c.get('dtype', 'bf16')]
    if kind == 'dense':
        w = [int(x) for x in c['widths'].split('-')]
        weights = sum(a * b for a, b in zip(w, w[1:]))
        return {'flops': 2.0 * c['batch'] * weights, 'bytes': es * (weights + sum(w[1:]) + c['batch'] * (w[0] + w[-1]))}
    if kind == 'backward':
        o = _out(c['hw'], c['stride'])
        x, f, g = c['n'] * c['hw'] ** 2 * c['ci'], c['k'] ** 2 * c['ci'] * c['co'], c['n'] * o * o * c['co']
        return {'flops': _backward_flops(c), 'bytes': es * (2 * x + 2 * f + g)}
    if kind == 'batched':
        b, r, k, d = c['batch'], c['rows'], c['cols'], c['d']
        return {'flops': 4.0 * b * r * k * d, 'bytes': es * b * (2 * r * d + 2 * k * d)}
    if kind == 'rows':
        n = c['rows'] * c['cols']
        out = {'mvn': n * es, 'softmax': n * es, 'topk': c['rows'] * min(10, c['cols']) * (es + 4), 'argmax': c['rows'] * 4}[c['op']]
        return {'flops': n, 'bytes': n * es + out}
    if kind == 'gemm':
        m, n, k = c['m'], c['n'], c['k']
        return {'flops': 2.0 * m * n * k, 'bytes': es * (m * k + k * n + m * n) + 4 * n}
    if kind == 'conv':
        o = _out(c['hw'], c['stride'])
        oes = 4 if c['dtype'] == 'i8' else es
        return {'flops': _conv_flops(c), 'bytes': es * (c['n'] * c['hw'] ** 2 * c['ci'] + c['k'] ** 2 * c['ci'] * c['co']) + oes * c['n'] * o * o * c['co']}
    px, o = c['n'] * c['hw'] ** 2, _out(c['hw'], 2)
    return {'flops': 2.0 * px * c['c'] * (9 + c['c']), 'bytes': 2 * (px * c['c'] + c['c'] * (c['c'] + 9 + 2)) + 6 * c['n'] * o * o * c['c']}


def tolerance(case):
    if case['kind'] == 'network':
        return {'rel': 1e-2}       # bf16 between fifty layers
    if case['kind'] == 'block':
        return {'rel': 1e-2, 'differ': 5e-3}  # window positions of near-equal bf16 values
    if case['kind'] == 'rows' and case['op'] in ('topk', 'argmax'):
        return 'exact'             # values and positions of given elements
    if case['dtype'] == 'i8':
        return 'exact'             # integer sums, one defined rounding
    if case['dtype'] == 'f32x3':
        return {'rel': 5e-5}       # 2^-16 a product
    if case['kind'] == 'backward' and case['dtype'] == 'f32':
        return {'rel': 3e-5}       # fp32 sums over every pixel of a batch
    return {'rel': 1e-5} if case['dtype'] == 'f32' else {'rel': 1e-2}


# ---- programs through Runner: host arrays in, host arrays out --------------------------------------------

class _Program:
    """A compiled program and the host arrays of one batch."""

    def __init__(self, program, inputs, staged=False):
        self.runner = P.Runner(program, target='hip')
        self.inputs = None if staged else inputs
        self.staged = self.runner.stage(inputs) if staged else None

    def run(self):
        if self.staged is not None:
            self.runner.run_staged(self.staged)
            return self.runner.fetch()
        return self.runner.run(self.inputs)


def _uniform(rng, shape, limit):
    return (rng.random(shape, dtype=np.float32) * 2 - 1) * np.float32(limit)


def _normal(rng, shape, scale=1.0):
    return rng.standard_normal(shape, dtype=np.float32) * np.float32(scale)


def _dtype(name):
    return {'f32': P.DType.FLOAT32, 'bf16': P.DType.BFLOAT16}[name]


def _network(c, seed):
    program, _, _ = resnet50.build(P, Pop, batch=c['batch'], round_fn=P.round_bf16, seed=12 + 100 * (seed % 1000))
    # Random weights without the scales of a trained network's folded normalisations let the activations double from
    # block to block; the image is scaled down so that the scores come out of order one, as a trained network's do.
    image = np.random.default_rng(seed).random((c['batch'], 224, 224, 3), dtype=np.float32) * np.float32(2.0 ** -11)
    return _Program(program, [image], staged=True)


def _dense(c, seed):
    rng, dt = np.random.default_rng(seed), _dtype(c['dtype'])
    widths = [int(x) for x in c['widths'].split('-')]
    X = P.Placeholder(dt, [c['batch'], widths[0]])
    x = X
    for a, b in zip(widths, widths[1:]):
        limit = math.sqrt(6.0 / (a + b))  # Glorot
        x = Pop.relu(Pop.dot(x, P.Constant(_uniform(rng, (a, b), limit), dt)) + P.Constant(_uniform(rng, (b,), 0.1), dt))
    return _Program(P.Program('dense', [X], [x]), [rng.random((c['batch'], widths[0]), dtype=np.float32)])


def _backward(c, seed):
    rng, dt = np.random.default_rng(seed), _dtype(c['dtype'])
    n, hw, ci, co, k, s = (c[x] for x in ('n', 'hw', 'ci', 'co', 'k', 'stride'))
    o = _out(hw, s)
    X, F, G = P.Placeholder(dt, [n, hw, hw, ci]), P.Placeholder(dt, [k, k, ci, co]), P.Placeholder(dt, [n, o, o, co])
    dX = Pop.convolution(G, F, strides=[s, s], deriv_mode=Pop.DERIV_DATA, result_shape=[hw, hw])
    dF = Pop.convolution(X, G, strides=[s, s], deriv_mode=Pop.DERIV_FILTER, result_shape=[k, k])
    inputs = [_normal(rng, (n, hw, hw, ci)), _normal(rng, (k, k, ci, co), math.sqrt(2.0 / (k * k * ci))), _normal(rng, (n, o, o, co))]
    return _Program(P.Program('conv_gradients', [X, F, G], [dX, dF]), inputs)


def _batched(c, seed):
    rng, dt = np.random.default_rng(seed), _dtype(c['dtype'])
    B, R, C, D = c['batch'], c['rows'], c['cols'], c['d']
    Q, K, V = P.Placeholder(dt, [B, R, D]), P.Placeholder(dt, [B, C, D]), P.Placeholder(dt, [B, C, D])
    b, i, j, d = P.TensorIndexes(4)
    S = P.Contraction().outShape(B, R, C).outAccess(b, i, j).sum(Q[b, i, d] * K[b, j, d]).build()
    W = Pop.softmax(S * (1.0 / math.sqrt(D)), -1)
    O = P.Contraction().outShape(B, R, D).outAccess(b, i, d).sum(W[b, i, j] * V[b, j, d]).build()
    return _Program(P.Program('batched', [Q, K, V], [O]), [_normal(rng, (B, R, D)), _normal(rng, (B, C, D)), _normal(rng, (B, C, D))])


def _rows(c, seed):
    rng, dt = np.random.default_rng(seed), _dtype(c['dtype'])
    R, C = c['rows'], c['cols']
    X = P.Placeholder(dt, [R, C])
    x = _normal(rng, (R, C))
    if c['op'] == 'mvn':
        g, s = P.Placeholder(dt, [C]), P.Placeholder(dt, [C])
        return _Program(P.Program('rows', [X, g, s], [Pop.mvn(X, axes=[1]) * g + s]), [x, 1 + _uniform(rng, C, 0.5), _uniform(rng, C, 0.5)])
    if c['op'] == 'softmax':
        outs = [Pop.softmax(X, -1)]
    elif c['op'] == 'topk':
        outs = list(Pop.topk(X, min(10, C)))
    else:
        outs = [Pop.argmax(X, 1)]
    return _Program(P.Program('rows', [X], outs), [x])


# ---- the kernel library on tensors that live on the GPU ---------------------------------------------------

HK = {'f32': hk.F32, 'f32x3': hk.F32, 'bf16': hk.BF16, 'i8': hk.I8}
TORCH = {'f32': torch.float32, 'f32x3': torch.float32, 'bf16': torch.bfloat16, 'i8': torch.int8}


class _Invokes:
    """Plans, the tensors their invokes read and write, and the invokes of one pass (arguments fixed, as in a serving loop)."""

    def __init__(self):
        hk.init(0)
        self.gen = torch.Generator(device='cuda')
        self.plans, self.keep, self.calls, self.outs = [], [], [], []

    def plan(self, family, desc):
        p = getattr(hk.lib(), 'pml_hip_%s_dispatch' % family)(ctypes.byref(desc))
        if not p:
            raise RuntimeError(hk.lib().pml_hip_last_error().decode())
        self.plans.append(p)
        return p

    def random(self, dtype, shape, scale=1.0):
        if dtype == 'i8':
            values = torch.randint(-127, 128, shape, generator=self.gen, device='cuda', dtype=torch.int8)
        else:
            values = torch.randn(shape, generator=self.gen, device='cuda') * scale
        return self.empty(TORCH[dtype], shape).copy_(values)

    def empty(self, dtype, shape):
        n = math.prod(shape)
        t = torch.empty(n + 64, dtype=dtype, device='cuda')[:n].view(shape)  # vector loads may end behind the last element
        self.keep.append(t)
        return t

    def operands(self, *tensors):
        return hk.ptr_array([t.data_ptr() for t in tensors])

    def call(self, name, *args):
        self.calls.append((getattr(hk.lib(), name), args + (None,)))  # the default stream

    def run(self):
        for fn, args in self.calls:
            hk.check(fn(*args))
        return self.outs

    def __del__(self):
        try:
            for p in self.plans:
                hk.lib().pml_hip_plan_free(p)
        except Exception:
            pass


def _gemm(c, seed):
    s = _Invokes()
    s.gen.manual_seed(seed)
    m, n, k, dtype = c['m'], c['n'], c['k'], c['dtype']
    g = hk.GemmDesc()
    g.in_dtype = HK[dtype]
    g.m, g.n, g.k, g.lda, g.ldc = m, n, k, k, n
    g.b_layout, g.ldb = (1, k) if c['b'] == 'nk' else (0, n)
    scale = 1.0 / math.sqrt(k)
    A, B = s.random(dtype, (m, k)), s.random(dtype, (n, k) if c['b'] == 'nk' else (k, n), scale)
    init = None
    if dtype == 'i8':  # cast to fp32, per-column scale, clamp, round, cast to int8
        g.out_dtype, g.c_dtype = hk.I32, hk.I8
        S = torch.empty(n, device='cuda').uniform_(0.001, 0.01, generator=s.gen) * (4.0 / math.sqrt(k))
        g.tail = hk.make_tail(ops=[(hk.EPI_CAST, hk.F32, 0, 0, 0.0), (hk.EPI_MUL, hk.F32, hk.OPND_TENSOR, 0, 0.0),
                                   (hk.EPI_MAX_GT, hk.F32, hk.OPND_IMM, 0, -127.0), (hk.EPI_MIN, hk.F32, hk.OPND_IMM, 0, 127.0),
                                   (hk.EPI_ROUND, hk.F32, 0, 0, 0.0), (hk.EPI_CAST, hk.I8, 0, 0, 0.0)], operands=[(hk.F32, 0, 1)])
        s.keep.append(S)
        ops, C = s.operands(S), s.empty(torch.int8, (m, n))
    else:
        g.out_dtype = g.c_dtype = HK[dtype]
        if dtype == 'f32x3':
            g.flags = hk.FP32_AS_BF16X3
        g.init_kind, g.init_dtype, g.init_row_stride, g.init_col_stride = 1, HK[dtype], 0, 1
        g.tail = hk.make_tail(ops=[(hk.EPI_RELU, HK[dtype], 0, 0, 0.0)])
        init = s.random(dtype, (n,), 0.1).data_ptr()
        ops, C = hk.ptr_array([]), s.empty(TORCH[dtype], (m, n))
    p = s.plan('gemm', g)
    b = B.data_ptr()
    if c['b'] == 'packed':
        hk.check(hk.lib().pml_hip_gemm_pack_b(p, b, None))
        b = None
    s.call('pml_hip_gemm_invoke', p, A.data_ptr(), b, C.data_ptr(), init, ops, hk.ptr_array([]))
    s.outs = [C]
    return s


def _conv(c, seed):
    s = _Invokes()
    s.gen.manual_seed(seed)
    n, hw, ci, co, k, st, dtype = (c[x] for x in ('n', 'hw', 'ci', 'co', 'k', 'stride', 'dtype'))
    o = _out(hw, st)
    d = hk.Conv2dDesc()
    d.in_dtype = HK[dtype]
    d.out_dtype = d.c_dtype = hk.I32 if dtype == 'i8' else HK[dtype]
    d.n, d.h, d.w, d.ci, d.kh, d.kw, d.co, d.oh, d.ow = n, hw, hw, ci, k, k, co, o, o
    d.stride_h = d.stride_w = st
    d.dil_h = d.dil_w = 1
    d.pad_h = d.pad_w = max(0, (o - 1) * st + k - hw) // 2
    init = None
    if dtype != 'i8':
        d.init_kind, d.init_dtype, d.init_row_stride, d.init_col_stride = 1, HK[dtype], 0, 1
        d.tail = hk.make_tail(ops=[(hk.EPI_RELU, HK[dtype], 0, 0, 0.0)])
        init = s.random(dtype, (co,), 0.1).data_ptr()
    X, F = s.random(dtype, (n, hw, hw, ci)), s.random(dtype, (k, k, ci, co), math.sqrt(2.0 / (k * k * ci)))
    O = s.empty(torch.int32 if dtype == 'i8' else TORCH[dtype], (n, o, o, co))
    p = s.plan('conv2d', d)
    f = F.data_ptr()
    if c['packed']:
        hk.check(hk.lib().pml_hip_conv2d_pack_filter(p, f, None))
        f = None
    none = hk.ptr_array([])
    s.call('pml_hip_conv2d_invoke', p, X.data_ptr(), f, O.data_ptr(), init, none, none)
    s.outs = [O]
    return s


def _block(c, seed):
    s = _Invokes()
    s.gen.manual_seed(seed)
    n, hw, ch = c['n'], c['hw'], c['c']
    px, o, none = n * hw * hw, _out(hw, 2), hk.ptr_array([])
    pitch = (ch * 2 + 127) // 128 * 64  # rows of whole 128-byte lines, as the planner lays such a temporary out
    I, D, R = s.random('bf16', (n, hw, hw, ch)), s.empty(torch.bfloat16, (px, pitch)), s.empty(torch.bfloat16, (n, hw, hw, ch))
    Fd, Fp = s.random('bf16', (3, 3, ch), math.sqrt(2.0 / 9)), s.random('bf16', (ch, ch), math.sqrt(2.0 / ch))
    scale, shift = s.random('bf16', (ch,), 0.2) + 1, s.random('bf16', (ch,), 0.2)
    s.keep.append(scale)
    M, X = s.empty(torch.bfloat16, (n, o, o, ch)), s.empty(torch.int32, (n, o, o, ch))
    d = hk.Dwconv2dDesc()
    d.dtype, d.out_pitch = hk.BF16, pitch
    d.n, d.h, d.w, d.c, d.kh, d.kw, d.oh, d.ow = n, hw, hw, ch, 3, 3, hw, hw
    d.stride_h = d.stride_w = d.dil_h = d.dil_w = d.pad_h = d.pad_w = 1
    pd = s.plan('dwconv2d', d)
    hk.check(hk.lib().pml_hip_dwconv2d_pack_filter(pd, Fd.data_ptr(), None))
    s.call('pml_hip_dwconv2d_invoke', pd, I.data_ptr(), None, D.data_ptr(), none, none)
    g = hk.GemmDesc()
    g.in_dtype = g.out_dtype = g.c_dtype = hk.BF16
    g.m, g.n, g.k, g.lda, g.ldb, g.ldc = px, ch, ch, pitch, ch, ch
    g.tail = hk.make_tail(ops=[(hk.EPI_MUL, hk.BF16, hk.OPND_TENSOR, 0, 0.0), (hk.EPI_ADD, hk.BF16, hk.OPND_TENSOR, 1, 0.0),
                               (hk.EPI_RELU, hk.BF16, 0, 0, 0.0)], operands=[(hk.BF16, 0, 1), (hk.BF16, 0, 1)])
    pg = s.plan('gemm', g)
    hk.check(hk.lib().pml_hip_gemm_pack_b(pg, Fp.data_ptr(), None))
    s.call('pml_hip_gemm_invoke', pg, D.data_ptr(), None, R.data_ptr(), None, s.operands(scale, shift), none)
    q = hk.Pool2dDesc()
    q.dtype, q.agg, q.with_index = hk.BF16, hk.AGG_MAX, 1
    q.n, q.h, q.w, q.c, q.kh, q.kw, q.oh, q.ow = n, hw, hw, ch, 3, 3, o, o
    q.stride_h = q.stride_w = 2
    q.pad_h = q.pad_w = max(0, (o - 1) * 2 + 3 - hw) // 2
    s.call('pml_hip_pool2d_invoke', s.plan('pool2d', q), R.data_ptr(), M.data_ptr(), X.data_ptr())
    s.outs = [M, X]
    return s


_PREPARE = {'network': _network, 'dense': _dense, 'backward': _backward, 'batched': _batched, 'rows': _rows, 'gemm': _gemm, 'conv': _conv,
            'block': _block}


def prepare(case, seed):
    return _PREPARE[case['kind']](case, seed)


def run(state):
    return state.run()
