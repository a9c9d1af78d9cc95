"""Performance cases: the work a program has this package do, through its public entry points.

`listed()` are fixed cases, `draw(rng)` gives further ones of the same ranges.  A case is a dict of plain values with
a `kind`; `prepare` makes what the program holds before the call, `run` is one pass.

kind       the pass
layer      one serving call of a layer with a frozen int8 weight, issued from Python
mlp_serve  `blocks` MLP blocks (d -> ff, ReLU, ff -> d) with frozen weights, recorded once and replayed
train      one quantized dot_general, forward and both gradients, stochastic rounding in the gradients
mlp_train  forward and backward of a float32 two-layer MLP block, recorded once and replayed with the key on the device
fp8_train  the attention projection 'bsd,dhk->bshk' in e4m3, gradients in e5m2 with stochastic rounding
tiled      a serving layer with a frozen int4 weight and one scale per 128 k of a row or column
ragged     the mixture-of-experts contraction, both operands quantized in the call
conv       a quantized convolution forward, recorded once and replayed
"""
import numpy as np
import torch

from aqt_amd.v2 import aqt_conv_general
from aqt_amd.v2 import aqt_dot_general as aqt
from aqt_amd.v2 import aqt_ragged_dot
from aqt_amd.v2 import config
from aqt_amd.v2 import hip_graph
from aqt_amd.v2 import tiled_dot_general
from aqt_amd.v2 import utils
from aqt_amd.v2.flax import aqt_flax

MATMUL = (((1,), (0,)), ((), ()))
GROUP = 128  # k per scale of the tiled layer


def listed():
  return [
      # the smallest call: one token of a decode loop through one projection, every launch issued from Python
      dict(name='layer_1_token', kind='layer', m=1, k=4096, n=4096),
      # a decode step of a small batch through the MLP blocks of two layers, int8 weights
      dict(name='mlp_8_tokens_int8', kind='mlp_serve', m=8, d=4096, ff=14336, blocks=2, bits=8, weight_only=False),
      # the same with int4 weights and a batch that is no round number
      dict(name='mlp_33_tokens_int4', kind='mlp_serve', m=33, d=4096, ff=11008, blocks=2, bits=4, weight_only=False),
      # prefill of a prompt of arbitrary length
      dict(name='mlp_1000_rows_int8', kind='mlp_serve', m=1000, d=4096, ff=14336, blocks=1, bits=8, weight_only=False),
      # the same with the activations left in bfloat16
      dict(name='mlp_500_rows_weight_only', kind='mlp_serve', m=500, d=4096, ff=14336, blocks=1, bits=8, weight_only=True),
      # training step of a layer whose sizes are no multiples of anything
      dict(name='train_odd_sizes', kind='train', m=1999, k=1030, n=3001, dtype='bf16'),
      # training step of the MLP projection of a large language model
      dict(name='train_large', kind='train', m=8192, k=4096, n=14336, dtype='bf16'),
      # training step of a small float32 network
      dict(name='mlp_train_f32', kind='mlp_train', rows=4096, d=512, hidden=2048),
      # training step of an attention projection in fp8
      dict(name='fp8_projection_train', kind='fp8_train', batch=8, seq=4096, d=4096, heads=32, head_dim=128),
      # prefill against a weight with subchannel scales
      dict(name='tiled_2048_rows_int4', kind='tiled', m=2048, k=8192, n=28672),
      # a mixture-of-experts layer
      dict(name='ragged_8_experts', kind='ragged', tokens=8192, experts=8, k=4096, n=14336),
      # a 3 x 3 convolution of an image network
      dict(name='conv_3x3', kind='conv', batch=32, size=56, cin=128, cout=128, window=3, stride=1),
  ]


def draw(rng):
  def log(lo, hi, step=1):
    """lo .. hi, spread over the logarithm, a multiple of step."""
    v = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(round(v / step)) * step))

  kind = rng.choice(['layer', 'mlp_serve', 'mlp_serve', 'mlp_serve', 'train', 'train', 'mlp_train', 'fp8_train', 'tiled',
                     'ragged', 'conv'])
  if kind == 'layer':
    return dict(kind=kind, m=log(1, 2048), k=log(512, 8192, 16), n=log(512, 14336, 16))
  if kind == 'mlp_serve':
    weight_only = rng.random() < 0.34
    return dict(kind=kind, m=log(1, 2048), d=log(1024, 4096, 32), ff=log(2048, 14336, 32), blocks=rng.choice([1, 2]),
                bits=rng.choice([4, 8]), weight_only=weight_only)
  if kind == 'train':
    step = rng.choice([1, 8, 64])
    return dict(kind=kind, m=log(128, 8192, step), k=log(128, 4096, step), n=log(128, 14336, step),
                dtype=rng.choice(['bf16', 'bf16', 'f32']))
  if kind == 'mlp_train':
    return dict(kind=kind, rows=log(256, 4096), d=log(128, 1024, 8), hidden=log(256, 4096, 8))
  if kind == 'fp8_train':
    return dict(kind=kind, batch=rng.choice([1, 2, 4, 8]), seq=log(128, 4096), d=log(512, 4096, 32),
                heads=rng.choice([4, 8, 16, 32]), head_dim=rng.choice([64, 128]))
  if kind == 'tiled':
    return dict(kind=kind, m=log(1, 2048), k=log(1024, 8192, GROUP), n=log(1024, 28672, 16))
  if kind == 'ragged':
    return dict(kind=kind, tokens=log(64, 8192), experts=rng.choice([4, 8, 16]), k=log(512, 4096, 16),
                n=log(512, 7168, 16))
  return dict(kind=kind, batch=log(1, 32), size=log(7, 56), cin=rng.choice([64, 96, 128, 256]),
              cout=rng.choice([64, 96, 128, 256]), window=rng.choice([1, 3, 3, 5]), stride=rng.choice([1, 1, 2]))


def _gen(seed):
  g = torch.Generator(device='cuda')
  g.manual_seed(seed)
  return g


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
  return (torch.randn(*shape, generator=g, device='cuda') * std).to(dtype)


def _activations(g, *shape, dtype=torch.bfloat16):
  """Unit normal, one value in 200 twenty times as large."""
  x = torch.randn(*shape, generator=g, device='cuda')
  return torch.where(torch.rand(*shape, generator=g, device='cuda') < 0.005, x * 20, x).to(dtype)


def _key(seed):
  return utils.prng_key(seed % (1 << 31))


def _frozen_layer(cfg, x, w, seed, tiling=None):
  """A serving layer whose weight was quantized once; what a program restores from its checkpoint."""
  freeze = aqt_flax.FreezerMode

  def make(mode):
    return aqt_flax.AqtDotGeneral(
        cfg, rhs_quant_mode=mode, tiling_cfg=tiling, use_legacy_freezer=False, lhs_freeze_mode=freeze.CALIBRATION,
        rhs_freeze_mode=freeze.CALIBRATION_AND_VALUE, rngs={'params': _key(seed)})

  convert = make(utils.QuantMode.CONVERT)
  convert(x, w, MATMUL, None)
  serve = make(utils.QuantMode.SERVE)
  serve.load_variables(convert.variables())
  return serve


def _serving_cfg(bits, weight_only):
  if weight_only:
    return aqt.dot_general_make(None, bits)
  return aqt.dot_general_make(8, bits)


def prepare(case, seed):
  g = _gen(seed)
  kind = case['kind']
  if kind == 'layer':
    m, k, n = case['m'], case['k'], case['n']
    x, w = _activations(g, m, k), _normal(g, k, n, std=0.02)
    with torch.no_grad():
      layer = _frozen_layer(_serving_cfg(8, False), x, w, seed)
      layer(x, w, MATMUL)
    return dict(kind=kind, layer=layer, x=x, w=w)
  if kind == 'mlp_serve':
    d, ff = case['d'], case['ff']
    cfg = _serving_cfg(case['bits'], case['weight_only'])
    x = _activations(g, case['m'], d)
    layers = []
    with torch.no_grad():
      for _ in range(case['blocks']):
        for k, n in ((d, ff), (ff, d)):
          w = _normal(g, k, n, std=k ** -0.5)
          layers.append((_frozen_layer(cfg, x if k == d else _activations(g, 4, ff), w, seed), w))

    def step(x):
      for i in range(0, len(layers), 2):
        (up, wu), (down, wd) = layers[i:i + 2]
        x = down(torch.relu(up(x, wu, MATMUL)), wd, MATMUL)
      return x

    # a recording reads the weights where they lie: the program keeps its layers
    return dict(kind=kind, step=hip_graph.GraphedCall(step, x), x=x, layers=layers)
  if kind == 'train':
    dt = {'bf16': torch.bfloat16, 'f32': torch.float32}[case['dtype']]
    m, k, n = case['m'], case['k'], case['n']
    lhs, rhs = _activations(g, m, k, dtype=dt).requires_grad_(True), _normal(g, k, n, std=0.02, dtype=dt).requires_grad_(True)
    cfg = config.set_context(config.fully_quantized(fwd_bits=8, bwd_bits=8), _key(seed), None)
    return dict(kind=kind, lhs=lhs, rhs=rhs, grad=_normal(g, m, n, std=1e-3, dtype=dt), cfg=cfg)
  if kind == 'mlp_train':
    rows, d, hidden = case['rows'], case['d'], case['hidden']
    x = _normal(g, rows, d, dtype=torch.float32).requires_grad_(True)
    w1 = _normal(g, d, hidden, std=d ** -0.5, dtype=torch.float32).requires_grad_(True)
    w2 = _normal(g, hidden, d, std=hidden ** -0.5, dtype=torch.float32).requires_grad_(True)
    grad = _normal(g, rows, d, std=1.0 / (rows * d), dtype=torch.float32)
    cfg = config.fully_quantized(fwd_bits=8, bwd_bits=8)
    keys = [torch.from_numpy(np.asarray(_key(seed + i), dtype=np.uint32).view(np.int32).copy()).cuda() for i in (1, 2)]

    def step():
      x.grad = w1.grad = w2.grad = None
      h = config.set_context(cfg, keys[0], None)(x, w1, MATMUL)
      y = config.set_context(cfg, keys[1], None)(torch.relu(h), w2, MATMUL)
      y.backward(grad)
      return y.detach(), x.grad, w1.grad, w2.grad

    return dict(kind=kind, step=hip_graph.GraphedStep(step), reads=(x, w1, w2, grad, keys))
  if kind == 'fp8_train':
    d, h, p = case['d'], case['heads'], case['head_dim']
    x = _activations(g, case['batch'], case['seq'], d).requires_grad_(True)
    w = _normal(g, d, h, p, std=0.02).requires_grad_(True)
    cfg = config.config_v4(fwd_bits='e4m3', dlhs_bits='e5m2', drhs_bits='e5m2')
    for raw in (cfg.fwd, cfg.dlhs, cfg.drhs):
      raw.dg_quantizer.lhs.calib_shared_axes = 'per_tensor'
      raw.dg_quantizer.rhs.calib_shared_axes = 'per_tensor'
    return dict(kind=kind, x=x, w=w, grad=_normal(g, case['batch'], case['seq'], h, p, std=1e-3),
                cfg=config.set_context(cfg, _key(seed), None))
  if kind == 'tiled':
    x, w = _activations(g, case['m'], case['k']), _normal(g, case['k'], case['n'], std=0.015)
    side = lambda axis: tiled_dot_general.TensorTiling([tiled_dot_general.AxisTiling(axis=axis, tile_size=GROUP)], [])
    with torch.no_grad():
      layer = _frozen_layer(aqt.dot_general_make(8, 4), x, w, seed, tiled_dot_general.Cfg(lhs=side(1), rhs=side(0)))
      layer(x, w, MATMUL)
    return dict(kind=kind, layer=layer, x=x, w=w)
  if kind == 'ragged':
    tokens, experts = case['tokens'], case['experts']
    x, w = _activations(g, tokens, case['k']), _normal(g, experts, case['k'], case['n'], std=0.02)
    # uneven loads: every token picks an expert, some experts being more popular than others
    weights = torch.rand(experts, generator=g, device='cuda') + 0.25
    picks = torch.multinomial(weights, tokens, replacement=True, generator=g)
    return dict(kind=kind, x=x, w=w, sizes=torch.bincount(picks, minlength=experts).to(torch.int32))
  assert kind == 'conv', kind
  x = _activations(g, case['batch'], case['size'], case['size'], case['cin'])
  kernel = _normal(g, case['window'], case['window'], case['cin'], case['cout'], std=0.05)
  conv = aqt_conv_general.make_conv_general_dilated(aqt_conv_general.conv_general_dilated_make(2, 8, 8))
  dn = aqt_conv_general.flax_conv_dimension_numbers(x.shape)
  stride = (case['stride'], case['stride'])
  return dict(kind=kind, x=x, kernel=kernel, step=hip_graph.GraphedCall(
      lambda a: conv(a, kernel, stride, 'SAME', dimension_numbers=dn), x))


def run(state):
  kind = state['kind']
  if kind in ('layer', 'tiled'):
    with torch.no_grad():
      return state['layer'](state['x'], state['w'], MATMUL)
  if kind in ('mlp_serve', 'conv'):
    return state['step'](state['x'])
  if kind == 'mlp_train':
    return state['step'].replay()
  if kind == 'train':
    lhs, rhs = state['lhs'], state['rhs']
    lhs.grad = rhs.grad = None
    out = state['cfg'](lhs, rhs, MATMUL)
    out.backward(state['grad'])
    return out.detach(), lhs.grad, rhs.grad
  if kind == 'fp8_train':
    x, w = state['x'], state['w']
    x.grad = w.grad = None
    out = aqt.einsum('bsd,dhk->bshk', x, w, state['cfg'])
    out.backward(state['grad'])
    return out.detach(), x.grad, w.grad
  assert kind == 'ragged', kind
  with torch.no_grad():
    return aqt_ragged_dot.ragged_dot(state['x'], state['w'], state['sizes'])


def work(case):
  """Each input read once, each output written once; the operations of the contractions."""
  kind = case['kind']
  if kind == 'layer':
    m, k, n = case['m'], case['k'], case['n']
    return dict(bytes=k * n + 4 * n + 2 * m * (k + n), flops=2 * m * k * n)
  if kind == 'mlp_serve':
    m, d, ff, blocks = case['m'], case['d'], case['ff'], case['blocks']
    weight = d * ff * case['bits'] // 8
    return dict(bytes=blocks * (2 * weight + 4 * (d + ff)) + 4 * m * d, flops=blocks * 4 * m * d * ff)
  if kind == 'train':
    m, k, n = case['m'], case['k'], case['n']
    size = 2 if case['dtype'] == 'bf16' else 4
    return dict(bytes=2 * size * (m * k + k * n + m * n), flops=6 * m * k * n)
  if kind == 'mlp_train':
    rows, d, hidden = case['rows'], case['d'], case['hidden']
    return dict(bytes=4 * (4 * rows * d + 4 * d * hidden), flops=12 * rows * d * hidden)
  if kind == 'fp8_train':
    m, k, n = case['batch'] * case['seq'], case['d'], case['heads'] * case['head_dim']
    return dict(bytes=4 * (m * k + k * n + m * n), flops=6 * m * k * n)
  if kind == 'tiled':
    m, k, n = case['m'], case['k'], case['n']
    return dict(bytes=k * n // 2 + 4 * n * (k // GROUP) + 2 * m * (k + n), flops=2 * m * k * n)
  if kind == 'ragged':
    t, e, k, n = case['tokens'], case['experts'], case['k'], case['n']
    return dict(bytes=2 * (t * k + e * k * n + t * n), flops=2 * t * k * n)
  b, cin, cout, window = case['batch'], case['cin'], case['cout'], case['window']
  out = -(-case['size'] // case['stride'])
  return dict(bytes=2 * (b * case['size'] ** 2 * cin + window ** 2 * cin * cout + b * out ** 2 * cout),
              flops=2 * b * out ** 2 * window ** 2 * cin * cout)


def tolerance(case):
  """Integer contractions have one right answer: their operands, sums and the roundings that follow are all pinned."""
  if case['kind'] == 'fp8_train':
    # float sums of fp8 products: the fp8 matrix instruction against sums with every product bit kept, 4e-4 apart
    return dict(rel=2e-3)
  if case['kind'] == 'mlp_serve' and case['weight_only']:
    # bfloat16 results of float32 sums in another order, through up to four layers: 1.3e-3 between two kernels
    return dict(rel=5e-3)
  return 'exact'
