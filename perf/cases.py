"""The measured workloads of the driving-model framework.

Every case is a dict of plain values; `prepare` makes what a program holds
before the call, `run` makes one pass through the package's public entry
points, `exact` computes the same outputs in 64 bits with plain torch, `work`
counts the bytes and operations the pass cannot do without and `tolerance`
says how far two correct implementations may differ.

Kinds of case:
  layernorm  chestnut.kernels.layernorm   (row LayerNorm, f16 or f32 out)
  gemv       chestnut.kernels.gemv        (weight-streaming product, bias, GELU)
  gemm       chestnut.kernels.gemm        (f32 out; B as [K][N] or [N][K])
  gemm_epi   chestnut.kernels.gemm_epi    (bias / ReLU / GELU to f16, residual add)
  attention  chestnut.kernels.attention   (non-causal, packed QK and V^T)
  warp       chestnut.kernels.warp_nv12   (two NV12 camera frames -> model input)
  pack       chestnut.kernels.frames_to_tensor (I420 frame -> 6 channels)
  frame      chestnut.Engine.run_frame    (a whole recurrent policy frame)
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'chestnut-on-pc_amd'))

from chestnut import Engine  # noqa: E402
from chestnut import kernels as K  # noqa: E402
from chestnut import spec as S  # noqa: E402


# ------------------------------------------------------------------ the cases --
def listed():
    return [
        # The smallest call: the LayerNorm of the `tiny` spec's 64 tokens.
        dict(name='layernorm_tiny', kind='layernorm', rows=64, d=128, f16=True),
        # The widest model's LayerNorm over a batch of token blocks (32 frames of 512 tokens).
        dict(name='layernorm_batch', kind='layernorm', rows=16384, d=2048, f16=True),
        # The temporal context product of the 1B model: weights pass once.
        dict(name='gemv_temporal', kind='gemv', rows=3072, K=12288, bias=True, act=1),
        # The context product of the 1B model, a ragged K (3072 + 200 + 4, padded to 8).
        dict(name='gemv_context', kind='gemv', rows=2048, K=3280, bias=True, act=0),
        # The benchmark's single GEMM, B as the caller holds it, [K][N].
        dict(name='gemm_kn', kind='gemm', M=1024, N=1024, K=6144, kn=True, bias=False),
        # A large product: eight frames' tokens through a square layer.
        dict(name='gemm_large', kind='gemm', M=4096, N=4096, K=4096, kn=False, bias=True),
        # The 1B block's MLP up-projection with its GELU epilogue.
        dict(name='mlp_up', kind='gemm_epi', M=512, N=8192, K=2048, epi=3, bias=True),
        # A small, ragged residual product (39M model widths, tokens not a tile multiple).
        dict(name='resid_ragged', kind='gemm_epi', M=200, N=520, K=2048, epi=4, bias=True),
        # The 1B block's attention.
        dict(name='attention_1b', kind='attention', T=512, heads=16, hd=128),
        # The openpilot input stage: both road-camera frames to the model input.
        dict(name='warp_road', kind='warp', w=1928, h=1208, stride=2048, y_height=1216, mw=512, mh=256,
             division='ieee'),
        # Whole recurrent frames from host memory: the 39M model ...
        dict(name='frame_39m', kind='frame', spec='driving_39m', stem='32,64,128,256,256', d=512, heads=8, hd=64,
             layers=4, ff=2048, temporal=1664),
        # ... and the 1B model, the benchmark's model.
        dict(name='frame_1b', kind='frame', spec='big_driving_1b', stem='32,64,128,256,512', d=2048, heads=16, hd=128,
             layers=20, ff=8192, temporal=3072),
    ]


FLOPS_MAX = 1.3e11     # below the largest listed product
ELEMS_MAX = 1 << 25    # elements of a drawn LayerNorm or GEMV matrix


def _log(rng, lo, hi, mult=1):
    """An integer of [lo, hi], uniform over its logarithm, a multiple of `mult`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(lo, min(hi, int(v) // mult * mult))


def draw(rng):
    kind = rng.choice(['layernorm', 'layernorm', 'gemv', 'gemv', 'gemm', 'gemm', 'gemm', 'gemm_epi', 'gemm_epi',
                       'gemm_epi', 'attention', 'attention', 'warp', 'pack', 'frame', 'frame'])
    if kind == 'layernorm':
        d = rng.choice([128, 256, 512, 1024, 2048])
        return dict(kind=kind, rows=_log(rng, 1, min(32768, ELEMS_MAX // d)), d=d, f16=rng.random() < 0.7)
    if kind == 'gemv':
        k = _log(rng, 64, 16384, 8)
        return dict(kind=kind, rows=_log(rng, 4, min(16384, ELEMS_MAX // k)), K=k, bias=rng.random() < 0.7,
                    act=rng.choice([0, 0, 1]))
    if kind in ('gemm', 'gemm_epi'):
        while True:
            m, n, k = _log(rng, 1, 4096), _log(rng, 8, 8192, 8), _log(rng, 64, 8192, 64)
            if 2.0 * m * n * k <= FLOPS_MAX:
                break
        if kind == 'gemm':
            return dict(kind=kind, M=m, N=n, K=k, kn=rng.random() < 0.5, bias=rng.random() < 0.5)
        return dict(kind=kind, M=m, N=n, K=k, epi=rng.choice([1, 2, 3, 4]), bias=rng.random() < 0.8)
    if kind == 'attention':
        return dict(kind=kind, T=64 * rng.randint(1, 8), heads=rng.randint(1, 24), hd=rng.choice([64, 128]))
    if kind == 'warp':
        w, h = 2 * rng.randint(320, 1024), 2 * rng.randint(240, 640)
        return dict(kind=kind, w=w, h=h, stride=w + 8 * rng.randint(0, 16), y_height=h + 2 * rng.randint(0, 8),
                    mw=4 * rng.randint(32, 256), mh=4 * rng.randint(32, 128), division=rng.choice(['ieee', 'rcp']))
    if kind == 'pack':
        return dict(kind=kind, H=4 * _log(rng, 16, 400), W=2 * _log(rng, 32, 1024))
    hd = rng.choice([64, 128])
    heads = rng.choice([h for h in (1, 2, 4, 8, 16) if 128 <= h * hd <= 1024])
    d = heads * hd
    t = rng.choice([64, 128, 256, 512])
    return dict(kind='frame', spec='', stem=f'{rng.choice([8, 16, 32])},32,64,{min(t, 256)},{t}', d=d, heads=heads,
                hd=hd, layers=rng.randint(1, 6), ff=rng.choice([2, 4]) * d, temporal=64 * rng.randint(4, 32))


# ------------------------------------------------------------------- inputs --
def _gen(seed):
    g = torch.Generator(device='cuda')
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, scale=1.0, dtype=torch.float32, shift=0.0):
    return (torch.randn(shape, generator=g, device='cuda') * scale + shift).to(dtype)


def _bytes(g, n):
    return torch.randint(0, 256, (n,), generator=g, device='cuda', dtype=torch.uint8)


def _inputs(c, seed):
    """The tensors of a single-kernel case: activations of unit scale (they
    come out of a LayerNorm), weights N(0, 0.02) as the models' are."""
    g = _gen(seed)
    kind = c['kind']
    if kind == 'layernorm':
        d = c['d']
        return dict(x=_normal(g, (c['rows'], d), 2.0, shift=0.5), g=_normal(g, (d,), 0.02, shift=1.0),
                    b=_normal(g, (d,), 0.02))
    if kind == 'gemv':
        return dict(W=_normal(g, (c['rows'], c['K']), 0.02, torch.float16),
                    x=torch.rand(c['K'], generator=g, device='cuda') * 2 - 1,
                    b=_normal(g, (c['rows'],), 0.02) if c['bias'] else None)
    if kind == 'gemm':
        return dict(A=_normal(g, (c['M'], c['K']), 1.0, torch.float16),
                    B=_normal(g, (c['K'], c['N']) if c['kn'] else (c['N'], c['K']), 0.02, torch.float16),
                    b=_normal(g, (c['N'],), 0.02) if c['bias'] else None)
    if kind == 'gemm_epi':
        return dict(A=_normal(g, (c['M'], c['K']), 1.0, torch.float16),
                    W=_normal(g, (c['N'], c['K']), 0.02, torch.float16),
                    b=_normal(g, (c['N'],), 0.02) if c['bias'] else None,
                    out=_normal(g, (c['M'], c['N'])) if c['epi'] == 4 else
                    torch.empty(c['M'], c['N'], dtype=torch.float16, device='cuda'))
    if kind == 'attention':
        d = c['heads'] * c['hd']
        return dict(qk=_normal(g, (c['T'], 2 * d), 1.0, torch.float16), vt=_normal(g, (d, c['T']), 1.0, torch.float16))
    if kind == 'warp':
        n = c['stride'] * c['y_height'] + (c['h'] // 2) * c['stride']
        r = np.random.default_rng(int(seed))
        tfm = []
        for _ in range(2):   # the model view inside the camera frame, slightly rolled and tilted
            sx, sy = c['w'] / c['mw'] * r.uniform(0.5, 0.9), c['h'] / c['mh'] * r.uniform(0.5, 0.9)
            tfm.append(torch.tensor([[sx, r.normal(0, 0.02), c['w'] * r.uniform(0.05, 0.1)],
                                     [r.normal(0, 0.02), sy, c['h'] * r.uniform(0.05, 0.1)],
                                     [r.normal(0, 1e-6), r.normal(0, 1e-6), 1.0]], dtype=torch.float32).cuda())
        return dict(f=_bytes(g, n), bf=_bytes(g, n), tfm=tfm[0], btfm=tfm[1])
    return dict(f=_bytes(g, c['H'] * 3 // 2 * c['W']).reshape(c['H'] * 3 // 2, c['W']))


HISTORY = 100   # frames run before the measured one: every queue is full


class _Weights:
    """Parameters of a spec made on demand from one pool of normal values: each
    tensor starts at a place of its own, and the pool's length shares no factor
    with any row length, so rows do not repeat each other."""

    def __init__(self, spec, seed):
        self.table = {p[0]: p for p in S.param_table(spec)}
        self.order = {n: i for i, n in enumerate(self.table)}
        self.seed = int(seed)
        self.pool = np.random.default_rng(self.seed).standard_normal(4194301, dtype=np.float32)
        self.pool16 = (self.pool * np.float32(0.02)).astype(np.float16)

    def __getitem__(self, name):
        _, shape, dtype, init, scale = self.table[name]
        n = int(np.prod(shape))
        at = (self.order[name] * 104729 + 7 * self.seed) % self.pool.size
        small = dtype == 'f16' and scale == 0.02
        src = self.pool16 if small else self.pool
        v = np.concatenate([src[at:at + n], np.resize(src, max(0, n - (src.size - at)))]).reshape(shape)
        if small:
            return v
        v = v * np.float32(scale) + np.float32(1.0 if init == 'one_normal' else 0.0)
        return v.astype(np.float16 if dtype == 'f16' else np.float32)


def _spec(c):
    base = S.get_spec(c['spec'] or 'tiny')
    return dict(base, name=c['spec'] or 'perf', stem=[int(v) for v in c['stem'].split(',')], d_model=c['d'],
                n_heads=c['heads'], head_dim=c['hd'], n_layers=c['layers'], d_ff=c['ff'], temporal_dim=c['temporal'])


def _clip(spec, seed):
    """Five camera views and HISTORY + 1 packed inputs (desire pulses, traffic
    convention, action time, features of earlier frames)."""
    r = np.random.default_rng([int(seed), 1])
    views = r.integers(0, 256, (5, 2, 6, spec['img_h'], spec['img_w']), dtype=np.uint8)
    packed = np.zeros((HISTORY + 1, 12 + spec['feat_len']), np.float32)
    packed[:, :8] = r.random((HISTORY + 1, 8)) < 0.02
    packed[:, 8] = 1.0
    packed[:, 10:12] = (0.2, 0.05)
    packed[:, 12:] = np.tanh(r.standard_normal((HISTORY + 1, spec['feat_len'])) * 0.5)
    return views, packed


def prepare(case, seed):
    if case['kind'] != 'frame':
        return dict(_inputs(case, seed), case=case)
    spec = _spec(case)
    eng = Engine(spec, weights=_Weights(spec, seed))
    views, packed = _clip(spec, seed)
    for i in range(HISTORY):
        eng.run_frame(views[i % 5], packed[i])
    return dict(case=case, eng=eng, view=views[HISTORY % 5], packed=packed[HISTORY].copy(),
                hidden=eng.out_slices['hidden_state'])


def run(state):
    c = state['case']
    kind = c['kind']
    if kind == 'layernorm':
        return K.layernorm(state['x'], state['g'], state['b'], out_f16=c['f16'])
    if kind == 'gemv':
        return K.gemv(state['W'], state['x'], state['b'], act=c['act'])
    if kind == 'gemm':
        return K.gemm(state['A'], state['B'], b_kn=c['kn'], bias=state['b'])
    if kind == 'gemm_epi':
        return K.gemm_epi(state['A'], state['W'], state['b'], c['epi'], state['out'])
    if kind == 'attention':
        return K.attention(state['qk'], state['vt'], c['heads'], c['hd'])
    if kind == 'warp':
        return K.warp_nv12(state['f'], state['bf'], state['tfm'], state['btfm'], c['w'], c['h'], c['stride'],
                           c['y_height'], c['mw'], c['mh'], division=c['division'])
    if kind == 'pack':
        return K.frames_to_tensor(state['f'])
    # one frame of the recurrent loop: the new hidden state is the next frame's prev_feat
    out = state['eng'].run_frame(state['view'], state['packed'])
    state['packed'][12:] = out[state['hidden']]
    return out


# -------------------------------------------------------------------- costs --
def work(case):
    c = case
    kind = c['kind']
    if kind == 'layernorm':
        n = c['rows'] * c['d']
        return dict(bytes=4 * n + (2 if c['f16'] else 4) * n + 8 * c['d'], flops=8 * n)
    if kind == 'gemv':
        return dict(bytes=2 * c['rows'] * c['K'] + 4 * c['K'] + (8 if c['bias'] else 4) * c['rows'],
                    flops=2 * c['rows'] * c['K'])
    if kind in ('gemm', 'gemm_epi'):
        m, n, k = c['M'], c['N'], c['K']
        out = 4 if kind == 'gemm' else 8 if c['epi'] == 4 else 2
        return dict(bytes=2 * (m * k + n * k) + out * m * n + (4 * n if c['bias'] else 0), flops=2 * m * n * k)
    if kind == 'attention':
        d = c['heads'] * c['hd']
        return dict(bytes=8 * c['T'] * d, flops=4 * c['T'] * c['T'] * d)
    if kind == 'warp':
        px = 2 * 6 * (c['mh'] // 2) * (c['mw'] // 2)   # one texel read and one written per output byte
        return dict(bytes=2 * px + 72, flops=18 * px)
    if kind == 'pack':
        return dict(bytes=3 * c['H'] * c['W'], flops=c['H'] * c['W'] // 2 * 3)
    s = _spec(c)
    t, d, f = s['stem'][-1], s['d_model'], s['d_ff']
    params = sum(int(np.prod(p[1])) * (2 if p[2] == 'f16' else 4) for p in S.param_table(s))
    flops = s['n_layers'] * (2.0 * t * d * (4 * d + 2 * f) + 4.0 * t * t * d)
    ci, hw = 6 * s['n_frames'], s['img_h'] * s['img_w']
    for co in s['stem']:
        hw //= 4
        flops += 2 * 2.0 * hw * co * 9 * ci
        ci = co
    flops += 2.0 * t * d * 2 * hw + 2.0 * s['temporal_dim'] * s['feat_hist'] * s['feat_len']
    # parameters, the two sampled image pairs, the sampled features, inputs and outputs
    io = 2 * 2 * 6 * s['img_h'] * s['img_w'] + 4 * s['feat_hist'] * s['feat_len'] + 4 * S.output_size(s)
    return dict(bytes=params + io, flops=flops)


# ------------------------------------------------------------------- bounds --
def tolerance(case):
    kind = case['kind']
    if kind in ('warp', 'pack'):
        return 'exact'
    # about four times the error measured against 64 bits
    if kind == 'layernorm':
        return dict(rel=1e-3) if case['f16'] else dict(rel=1e-6)     # f16 rounding; f32 statistics
    if kind == 'gemv':
        return dict(rel=1e-6)                                       # f32 sums
    if kind == 'gemm' or (kind == 'gemm_epi' and case['epi'] == 4):
        return dict(rel=1.5e-6)                                     # f32 sums of exact f16 products
    if kind == 'gemm_epi':
        return dict(rel=1e-3)                                       # one f16 rounding
    if kind == 'attention':
        return dict(rel=1.2e-3)                                     # f16 probabilities and outputs
    return dict(rel=1e-3)                                           # f16 activations through every layer


# -------------------------------------------------------------------- exact --
def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _ln(x, g, b, eps=1e-5):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + eps) * g + b


def exact(case, seed):
    c = case
    kind = c['kind']
    if kind in ('warp', 'pack'):
        return None   # bytes that are moved, not computed
    if kind == 'frame':
        return _exact_frame(c, seed)
    s = {k: (v.double() if isinstance(v, torch.Tensor) else v) for k, v in _inputs(c, seed).items()}
    if kind == 'layernorm':
        return _ln(s['x'], s['g'], s['b'])
    if kind == 'gemv':
        y = s['W'] @ s['x']
        y = y + s['b'] if s['b'] is not None else y
        return _gelu(y) if c['act'] else y
    if kind == 'gemm':
        y = s['A'] @ (s['B'] if c['kn'] else s['B'].t().contiguous())
        return y + s['b'] if s['b'] is not None else y
    if kind == 'gemm_epi':
        y = s['A'] @ s['W'].t().contiguous()
        y = y + s['b'] if s['b'] is not None else y
        return {1: lambda: y, 2: lambda: y.clamp_min(0), 3: lambda: _gelu(y), 4: lambda: s['out'] + y}[c['epi']]()
    t, h, hd = c['T'], c['heads'], c['hd']
    return _attend(s['qk'][:, :h * hd], s['qk'][:, h * hd:], s['vt'].t(), t, h, hd)


def _attend(q, k, v, t, h, hd):
    o = torch.empty(t, h * hd, dtype=torch.float64, device=q.device)
    for i in range(h):
        sl = slice(i * hd, (i + 1) * hd)
        p = torch.softmax(q[:, sl].contiguous() @ k[:, sl].t().contiguous() / math.sqrt(hd), -1)
        o[:, sl] = p @ v[:, sl].contiguous()
    return o


def _exact_frame(c, seed):
    """The frame after HISTORY others, in 64 bits throughout (the engine's
    network as chestnut/spec.py lays it down)."""
    s = _spec(c)
    w = _Weights(s, seed)
    views, packed = _clip(s, seed)
    n, fs = HISTORY, s['frame_skip']

    def p(name):
        return torch.from_numpy(np.ascontiguousarray(w[name])).cuda().double()

    toks = []
    for b in range(2):
        x = np.concatenate([views[(n - fs) % 5][b], views[n % 5][b]])
        x = (torch.from_numpy(x).cuda().double() - 128.0) / 128.0
        for i in range(len(s['stem'])):
            wt = p(f'stem.{i}.w')[b].permute(0, 3, 1, 2).contiguous()
            cols = torch.nn.functional.unfold(x[None], 3, padding=1, stride=2)[0]
            y = wt.reshape(wt.shape[0], -1) @ cols + p(f'stem.{i}.b')[b][:, None]
            x = y.clamp_min(0).reshape(-1, (x.shape[1] + 1) // 2, (x.shape[2] + 1) // 2)
        toks.append(x.reshape(x.shape[0], -1))
    tok = torch.cat(toks, 1)
    pk = torch.from_numpy(packed).cuda().double()
    fl = fs * s['feat_hist']
    feat = torch.cat([pk[n - (fl - 1) + fs * k, 12:] for k in range(s['feat_hist'])])
    dl = fs * s['desire_hist']
    des = pk[[max(0, n - (dl - 1) + j) for j in range(dl)], :8].reshape(s['desire_hist'], fs, 8).amax(1).reshape(-1)
    tmp = _gelu(p('tmp.w') @ feat + p('tmp.b'))
    ctx = p('ctx.w') @ torch.cat([tmp, des, pk[n, 8:12]]) + p('ctx.b')
    x = tok @ p('emb.w').t().contiguous() + p('emb.b') + p('pos') + ctx
    t, d = x.shape
    for layer in range(s['n_layers']):
        q = f'blk.{layer}.'
        h = _ln(x, p(q + 'ln1.g'), p(q + 'ln1.b'))
        qkv = h @ p(q + 'qkv.w').t().contiguous() + p(q + 'qkv.b')
        a = _attend(qkv[:, :d], qkv[:, d:2 * d], qkv[:, 2 * d:], t, s['n_heads'], s['head_dim'])
        x = x + a @ p(q + 'o.w').t().contiguous() + p(q + 'o.b')
        h = _ln(x, p(q + 'ln2.g'), p(q + 'ln2.b'))
        u = _gelu(h @ p(q + 'up.w').t().contiguous() + p(q + 'up.b'))
        x = x + u @ p(q + 'down.w').t().contiguous() + p(q + 'down.b')
    pooled = _ln(x, p('lnf.g'), p('lnf.b')).mean(0)
    hp = pk[n, 12:]
    gi, gh = p('gru.wih') @ pooled + p('gru.bih'), p('gru.whh') @ hp + p('gru.bhh')
    hh = s['hidden']
    r, z = torch.sigmoid(gi[:hh] + gh[:hh]), torch.sigmoid(gi[hh:2 * hh] + gh[hh:2 * hh])
    nn = torch.tanh(gi[2 * hh:] + r * gh[2 * hh:])
    hid = (1 - z) * nn + z * hp
    return torch.cat([p('head.w') @ hid + p('head.b'), hid]).cpu()
