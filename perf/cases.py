"""Performance cases of dinosaur_amd: the work that its users have it do.

Five kinds of work, each through the package's public entry points:

* ``transform``: ``Grid.to_nodal`` and ``Grid.to_modal`` of a batch of fields,
  optionally with the gradient through both (data processing, losses, and
  the parity runs in float64);
* ``winds``: ``vor_div_to_uv_nodal`` and ``uv_nodal_to_vor_div_modal`` (model
  output, initialisation from reanalysis winds);
* ``explicit``: one ``PrimitiveEquations.explicit_terms`` evaluation (a model
  that calls the dynamical core's tendencies from its own stepper);
* ``step``: ``imex_rk_sil3`` steps with ``exponential_step_filter`` (forecasts);
* ``adjoint``: a checkpointed rollout and the gradient of its loss with respect
  to the initial state (data assimilation, training).

Grids are the package's own truncations (``Grid.T21`` ... ``Grid.TL639``) and
``Grid.with_wavenumbers`` grids, whose 2M+1 or 3M+1 longitudes are whatever
they are.  Inputs are developed-flow-like spectra; every field has the size it
has in the atmosphere.  ``exact`` restates the same computations with dense
float64 tensor operations.
"""
import functools
import math

import numpy as np
import torch

from dinosaur_amd import coordinate_systems
from dinosaur_amd import held_suarez
from dinosaur_amd import primitive_equations
from dinosaur_amd import sigma_coordinates
from dinosaur_amd import spherical_harmonic
from dinosaur_amd import time_integration
from dinosaur_amd import units as units_lib

DEVICE = 'cuda'
FIELDS = ('vorticity', 'divergence', 'temperature_variation', 'log_surface_pressure')
TRACERS = ('specific_humidity', 'specific_cloud_liquid_water_content',
           'specific_cloud_ice_water_content')
REFERENCE_TEMPERATURE = 288.0
VORTICITY_WEIGHT = 100.0  # of the loss: 0.05 of vorticity counts as 0.5 K

# truncation -> (max wavenumber, Gaussian nodes per quarter circle), Grid.construct
GRIDS = {
    'T21': (21, 16), 'T31': (31, 24), 'T42': (42, 32), 'T85': (85, 64), 'T106': (106, 80),
    'T119': (119, 90), 'T170': (170, 128), 'T213': (213, 160), 'T340': (340, 256),
    'T425': (425, 320), 'TL31': (31, 16), 'TL47': (47, 24), 'TL63': (63, 32), 'TL95': (95, 48),
    'TL127': (127, 64), 'TL159': (159, 80), 'TL179': (179, 90), 'TL255': (255, 128),
    'TL639': (639, 320),
}


def listed():
  return [
      # a small interactive run: one dry field set on the smallest grid
      dict(name='transform_T21_12', kind='transform', grid='T21', dtype='float32',
           precision='float32', fields=12, gradient=False),
      # the isolated transform round trip: 37 levels x 6 fields
      dict(name='transform_TL255_222', kind='transform', grid='TL255', dtype='float32',
           precision='float32', fields=222, gradient=False),
      # a spectral loss on three model fields, forward and backward, 320 x 160 nodes
      dict(name='gradient_T106_111', kind='transform', grid='T106', dtype='float32',
           precision='float32', fields=111, gradient=True),
      # float64, the precision in which results are compared with other models
      dict(name='transform_T85_f64_96', kind='transform', grid='T85', dtype='float64',
           precision='float32', fields=96, gradient=False),
      # one field on 37 levels at the resolution of operational analyses
      dict(name='transform_TL639_37', kind='transform', grid='TL639', dtype='float32',
           precision='float32', fields=37, gradient=False),
      # split-BF16 arithmetic on a quadratic grid of odd size, 268 x 134 nodes
      dict(name='transform_bf16x3_odd_64', kind='transform', grid='quadratic89',
           dtype='float32', precision='bf16x3', fields=64, gradient=False),
      # winds in and out of the model, 37 levels, 320 x 160 nodes
      dict(name='winds_TL159_37', kind='winds', grid='TL159', dtype='float32', layers=37),
      # tendencies of a single dry state for a caller's own stepper, 128 x 64 nodes
      dict(name='explicit_T42_L24', kind='explicit', grid='T42', dtype='float32', layers=24,
           moist=False, members=1),
      # a day of the small dry model advances 72 of these
      dict(name='step_T21_L12', kind='step', grid='T21', dtype='float32', layers=12, moist=False,
           held_suarez=False, members=1, steps=1, minutes=20),
      # one tick of a moist ensemble's largest group
      dict(name='step_T85_L24_moist_32', kind='step', grid='T85', dtype='float32', layers=24,
           moist=True, held_suarez=False, members=32, steps=1, minutes=10),
      # differentiable Held-Suarez rollout, one checkpoint segment of two steps
      dict(name='adjoint_TL127_L32', kind='adjoint', grid='TL127', dtype='float32', layers=32,
           moist=False, held_suarez=True, members=1, steps=2, minutes=10),
      # the full moist model: forward and checkpointed adjoint of 16 members
      dict(name='adjoint_TL255_L37_moist_16', kind='adjoint', grid='TL255', dtype='float32',
           layers=37, moist=True, held_suarez=False, members=16, steps=1, minutes=5),
  ]


def _log_int(rng, low, high):
  return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
  kind = rng.choice(['transform', 'transform', 'transform', 'winds', 'explicit', 'step',
                     'adjoint'])
  dtype = rng.choice(['float32', 'float32', 'float32', 'float64'])
  if kind in ('transform', 'winds'):
    if rng.random() < 0.3:
      grid = '%s%d' % (rng.choice(['quadratic', 'linear']), _log_int(rng, 21, 170))
    else:
      grid = rng.choice(sorted(GRIDS))
    _, _, I, J = _shape(grid)
    # at most the nodes of 300 fields on 512 x 256 in float32
    most = int(300 * 512 * 256 / (I * J) / (2 if dtype == 'float64' else 1))
    if kind == 'winds':
      return dict(kind=kind, grid=grid, dtype=dtype, layers=_log_int(rng, 1, min(137, most // 2)))
    gradient = rng.random() < 0.4
    precision = 'bf16x3' if dtype == 'float32' and rng.random() < 0.2 else 'float32'
    return dict(kind=kind, grid=grid, dtype=dtype, precision=precision,
                fields=_log_int(rng, 1, min(1000, most // (2 if gradient else 1))),
                gradient=gradient)
  grid = rng.choice(['T21', 'T31', 'T42', 'T85', 'T106', 'T119', 'T170', 'TL31', 'TL47', 'TL63',
                     'TL95', 'TL127', 'TL159', 'TL179', 'TL255'])
  _, _, I, J = _shape(grid)
  layers = rng.randint(8, 40)
  moist = rng.random() < 0.5
  # at most the nodes of one moist 37-level member on 512 x 256 (two in a forecast)
  budget = 37 * 512 * 256 * (1 if dtype == 'float64' or kind == 'adjoint' else 2)
  members = max(1, min(16, budget // (layers * I * J)))
  case = dict(kind=kind, grid=grid, dtype=dtype, layers=layers, moist=moist,
              members=_log_int(rng, 1, members))
  if kind == 'explicit':
    return case
  minutes = 1200 // _shape(grid)[0] if _shape(grid)[0] < 400 else 3
  return dict(case, held_suarez=not moist and rng.random() < 0.5, steps=rng.randint(1, 2),
              minutes=max(3, min(20, minutes)))


# ------------------------------------------------------------------ sizes


def _shape(name):
  """(M, L, I, J) of a grid name."""
  if name in GRIDS:
    n, g = GRIDS[name]
    return n + 1, n + 2, 4 * g, 2 * g
  for word, order in (('quadratic', 3), ('linear', 2)):
    if name.startswith(word):
      m = int(name[len(word):])
      nodes = order * m + 1
      return m, m + 1, nodes, (nodes + 1) // 2
  raise ValueError(name)


def _grid(name, precision='float32'):
  impl = functools.partial(spherical_harmonic.RealSphericalHarmonics,
                           transform_precision=precision)
  M, L, I, J = _shape(name)
  return spherical_harmonic.Grid(M, L, I, J, spherical_harmonics_impl=impl)


def _triangle(name):
  M, L, _, _ = _shape(name)
  return sum((1 if m == 0 else 2) * (L - m) for m in range(M))


def _transform_flops(name):
  """Of one field in one direction: the equatorially folded Legendre sums over
  the triangle and a real FFT of every latitude."""
  _, _, I, J = _shape(name)
  return J * _triangle(name) + 2.5 * I * math.log2(I) * J


def work(case):
  es = 8 if case['dtype'] == 'float64' else 4
  M, L, I, J = _shape(case['grid'])
  tri, flops = _triangle(case['grid']), _transform_flops(case['grid'])
  if case['kind'] == 'transform':
    passes = 2 if case['gradient'] else 1
    # round trip: modal in, nodal out, modal out; backward: two cotangents in, one out
    per_field = 2 * tri + I * J if passes == 1 else 4 * tri + 2 * I * J
    return {'bytes': es * case['fields'] * per_field, 'flops': 2 * passes * case['fields'] * flops}
  if case['kind'] == 'winds':
    return {'bytes': es * case['layers'] * (4 * tri + 2 * I * J),
            'flops': 4 * case['layers'] * flops}
  K, nt, E = case['layers'], len(TRACERS) if case['moist'] else 0, case['members']
  state = es * E * tri * ((3 + nt) * K + 1)
  inverse = (5 + nt) * K + 2 + (2 * K + 1 if case['moist'] else 0)
  forward = 6 * K + 1 + 3 * nt * K + (2 * K if case['moist'] else 0)
  if case.get('held_suarez'):
    inverse, forward = inverse + 3 * K + 1, forward + 3 * K
  evaluation = E * (inverse + forward) * flops
  if case['kind'] == 'explicit':
    return {'bytes': 2 * state, 'flops': evaluation}
  # three explicit evaluations a step; a gradient costs twice as much again
  passes = 1 if case['kind'] == 'step' else 3
  return {'bytes': (2 if passes == 1 else 4) * state,
          'flops': 3 * passes * case['steps'] * evaluation}


def tolerance(case):
  """About four times the error that the paths show against ``exact`` (2-norm, the
  worst output over the declared ranges; the winds' divergence is a small
  difference of large terms)."""
  if case['dtype'] == 'float64':
    return {'rel': {'transform': 1e-13, 'winds': 1e-12, 'explicit': 6e-13, 'step': 1e-13,
                    'adjoint': 2e-13}[case['kind']]}
  if case.get('precision') == 'bf16x3':
    return {'rel': 2e-5}
  return {'rel': {'transform': 4e-6, 'winds': 4e-4, 'explicit': 2.5e-5, 'step': 5e-6,
                  'adjoint': 1.4e-5}[case['kind']]}


# ------------------------------------------------------------------ inputs


def _noise(shape, gen):
  return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float64)


def _spectral(name, lead, gen, slope, first=1):
  """Gaussian coefficients on the triangle, falling as l**-slope from l = first."""
  M, L, _, _ = _shape(name)
  m = torch.arange(1, 2 * M, device=DEVICE) // 2
  l = torch.arange(L, device=DEVICE)
  amplitude = torch.where(l >= first, l.clamp(min=1).double() ** -slope, 0.0)
  return _noise(tuple(lead) + (2 * M - 1, L), gen) * (l >= m[:, None]) * amplitude


def _smooth_in_height(x, K):
  """Correlates neighbouring levels (x: (..., K, R, L)) as the atmosphere's are."""
  shift = min(3, K - 1)
  return (x + torch.roll(x, shift, -3)) / math.sqrt(2.0)


def _p0():
  return units_lib.SimUnits.from_si().nondimensionalize(1e5 * units_lib.scales.units.pascal)


def _state_arrays(case, seed):
  """Float64 coefficient arrays of one state: vorticity rms of a few 1e-5 / s,
  a tenth of it in the divergence, some kelvin of temperature variation,
  humidity decaying with height."""
  gen = torch.Generator(device=DEVICE).manual_seed(seed)
  name, K, E = case['grid'], case['layers'], case['members']
  lead = ((E,) if E > 1 else ()) + (K,)
  field = lambda slope: _smooth_in_height(_spectral(name, lead, gen, slope), K)  # noqa: E731
  out = {
      'vorticity': 0.15 * field(1.0),
      'divergence': 0.015 * field(1.0),
      'temperature_variation': 12.0 * field(1.5),
      'log_surface_pressure': 0.02 * _spectral(name, lead[:-1] + (1,), gen, 2.0),
  }
  root = math.sqrt(4 * math.pi)
  out['log_surface_pressure'][..., 0, 0] = root * math.log(_p0())
  if case['moist']:
    sigma = (torch.arange(K, device=DEVICE, dtype=torch.float64) + 0.5) / K
    profile = (sigma ** 3)[:, None, None]
    for tracer, mean in zip(TRACERS, (8e-3, 2e-5, 1e-5)):
      x = 0.5 * mean * field(1.5)
      x[..., 0, 0] += root * mean
      out[tracer] = x * profile
  return out


def _orography(name, seed):
  """Spectral coefficients of hills of some hundred metres, in Earth radii."""
  gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
  L = _shape(name)[1]
  x = _spectral(name, (), gen, 1.0) * 2e-4
  x[..., L - 1] = 0
  return x


def _targets(case, seed, shape):
  """Of the loss: nodal fields to compare the temperature and vorticity with."""
  gen = torch.Generator(device=DEVICE).manual_seed(seed + 2)
  return 0.5 * _noise(shape, gen), 0.05 * _noise(shape, gen)


def _dtype(case):
  return getattr(torch, case['dtype'])


def _time_step(case):
  return units_lib.SimUnits.from_si().nondimensionalize(
      60.0 * case['minutes'] * units_lib.scales.units.s)


def _model(case, seed):
  """(equation, Held-Suarez forcing or None, coords)."""
  specs = units_lib.SimUnits.from_si()
  coords = coordinate_systems.CoordinateSystem(
      _grid(case['grid']), sigma_coordinates.SigmaCoordinates.equidistant(case['layers']))
  moisture = dict(humidity_key=TRACERS[0], cloud_keys=TRACERS[1:]) if case['moist'] else {}
  reference = np.full(case['layers'], REFERENCE_TEMPERATURE)
  equation = primitive_equations.PrimitiveEquationsSigma(
      reference, _orography(case['grid'], seed).to(_dtype(case)), coords, specs, **moisture)
  forcing = None
  if case.get('held_suarez'):
    forcing = held_suarez.HeldSuarezForcingSigma(coords, specs, reference)
  return equation, forcing, coords


def _names(case):
  return FIELDS + (TRACERS if case.get('moist') else ())


def _state(leaves):
  return primitive_equations.State(
      *[leaves[f] for f in FIELDS], tracers={k: v for k, v in leaves.items() if k in TRACERS})


def _leaves(state):
  return {**{f: getattr(state, f) for f in FIELDS}, **state.tracers}


def _transform_inputs(case, seed):
  """Modal fields falling as l**-1.5 and, for a gradient, both cotangents."""
  gen = torch.Generator(device=DEVICE).manual_seed(seed)
  M, L, I, J = _shape(case['grid'])
  B = case['fields']
  x = [_spectral(case['grid'], (B,), gen, 1.5, first=0)]
  if case['gradient']:
    x += [_noise((B, I, J), gen), _spectral(case['grid'], (B,), gen, 0.0, first=0)]
  return [t.to(_dtype(case)) for t in x]


def _wind_inputs(case, seed):
  gen = torch.Generator(device=DEVICE).manual_seed(seed)
  lead = (case['layers'],)
  return [(0.15 * _spectral(case['grid'], lead, gen, 1.0)).to(_dtype(case)),
          (0.015 * _spectral(case['grid'], lead, gen, 1.0)).to(_dtype(case))]


def prepare(case, seed):
  if case['kind'] == 'transform':
    inputs = _transform_inputs(case, seed)
    inputs[0].requires_grad_(case['gradient'])
    return dict(case=case, grid=_grid(case['grid'], case['precision']), inputs=inputs)
  if case['kind'] == 'winds':
    return dict(case=case, grid=_grid(case['grid']), inputs=_wind_inputs(case, seed))
  leaves = {k: v.to(_dtype(case)).requires_grad_(case['kind'] == 'adjoint')
            for k, v in _state_arrays(case, seed).items()}
  equation, forcing, coords = _model(case, seed)
  state = dict(case=case, leaves=leaves, equation=equation, grid=coords.horizontal)
  if case['kind'] != 'explicit':
    dt = _time_step(case)
    composed = time_integration.compose_equations([equation, forcing]) if forcing else equation
    state['step'] = time_integration.step_with_filters(
        time_integration.imex_rk_sil3(composed, dt),
        [time_integration.exponential_step_filter(coords.horizontal, dt)])
  if case['kind'] == 'adjoint':
    shape = leaves['vorticity'].shape[:-3] + coords.horizontal.nodal_shape
    state['targets'] = [t.to(_dtype(case)) for t in _targets(case, seed, shape)]
  return state


# ------------------------------------------------------------------ one pass


def _loss(to_nodal, leaves, targets, layers):
  level = layers // 2
  t = to_nodal(leaves['temperature_variation'][..., level, :, :])
  z = to_nodal(leaves['vorticity'][..., level, :, :])
  return (((t - targets[0]) ** 2).mean() + VORTICITY_WEIGHT * ((z - targets[1]) ** 2).mean())


def run(state):
  case, grid = state['case'], state['grid']
  if case['kind'] == 'transform':
    x = state['inputs'][0]
    nodal = grid.to_nodal(x)
    modal = grid.to_modal(nodal)
    if not case['gradient']:
      return [nodal, modal]
    (gradient,) = torch.autograd.grad([nodal, modal], x, state['inputs'][1:])
    return [nodal.detach(), modal.detach(), gradient]
  if case['kind'] == 'winds':
    u, v = spherical_harmonic.vor_div_to_uv_nodal(grid, *state['inputs'])
    return [u, v, *spherical_harmonic.uv_nodal_to_vor_div_modal(grid, u, v)]
  if case['kind'] == 'explicit':
    with torch.no_grad():
      return _leaves(state['equation'].explicit_terms(_state(state['leaves'])))
  if case['kind'] == 'step':
    with torch.no_grad():
      x = _state(state['leaves'])
      for _ in range(case['steps']):
        x = state['step'](x)
      return _leaves(x)
  final = time_integration.checkpointed_rollout(state['step'], _state(state['leaves']),
                                                case['steps'], checkpoint_every=case['steps'])
  final = _leaves(final)
  loss = _loss(grid.to_nodal, final, state['targets'], case['layers'])
  names = _names(case)
  gradients = torch.autograd.grad(loss, [state['leaves'][k] for k in names])
  return dict(loss=loss.detach(), state={k: final[k].detach() for k in names},
              gradients=dict(zip(names, gradients)))


# ------------------------------------------------------------------ float64 restatement


def _gauss(n):
  """Gauss-Legendre nodes and weights, polished in extended precision."""
  x = np.polynomial.legendre.leggauss(n)[0].astype(np.longdouble)
  for _ in range(3):
    below, p = np.ones_like(x), x
    for l in range(2, n + 1):
      below, p = p, ((2 * l - 1) * x * p - (l - 1) * below) / l
    slope = n * (x * p - below) / (x * x - 1)
    x = x - p / slope
  return x.astype(np.float64), (2 / ((1 - x * x) * slope ** 2)).astype(np.float64)


class _Sphere:
  """Dense float64 transforms and spectral operators of one grid."""

  def __init__(self, name):
    self.M, self.L, self.I, self.J = M, L, I, J = _shape(name)
    x, w = _gauss(J)
    tensor = lambda a: torch.as_tensor(a, dtype=torch.float64, device=DEVICE)  # noqa: E731
    self.sin_lat = tensor(x)
    self.cos2 = 1 - self.sin_lat ** 2
    self.weights = tensor(2 * np.pi / I * w)
    # P[m, j, l] by the three-term recurrence from the sectoral values
    m = torch.arange(M, device=DEVICE, dtype=torch.float64)
    factors = torch.cat([tensor([math.sqrt(0.5)]), -torch.sqrt(1 + 0.5 / m[1:])])
    base = torch.where(m[:, None] > 0, torch.sqrt(self.cos2), 1.0) * factors[:, None]
    sectoral = torch.cumprod(base, 0)
    self.P = torch.zeros((M, J, L), dtype=torch.float64, device=DEVICE)
    below = torch.zeros((M, J), dtype=torch.float64, device=DEVICE)
    current = torch.zeros_like(below)
    eps = lambda l: torch.sqrt(  # noqa: E731
        ((l * l - m * m).clamp(min=0) / max(4.0 * l * l - 1, 1e-300)))[:, None]
    for l in range(L):
      if l:
        e1, e0 = eps(float(l)), eps(float(l - 1))
        nxt = torch.where(e1 > 0, (self.sin_lat * current - e0 * below) / e1.clamp(min=1e-300), 0)
        below, current = current, nxt
      if l < M:
        current = current.clone()
        current[l] = sectoral[l]
        below = below.clone()
        below[l] = 0
      self.P[:, :, l] = current
    angle = 2 * np.pi / I * ((np.arange(I)[:, None] * np.arange(M)[None]) % I)
    basis = np.stack([np.cos(angle), np.sin(angle)], -1) / np.sqrt(np.pi)
    basis[:, 0] = np.array([1 / np.sqrt(2 * np.pi), 0.0])
    self.F = tensor(basis.reshape(I, 2 * M))
    rows = np.arange(1, 2 * M) // 2
    l = np.arange(L)
    inside = l >= rows[:, None]
    lead = np.sqrt(np.where(inside, l ** 2 - rows[:, None] ** 2, 0) / np.maximum(4.0 * l ** 2 - 1, 1))
    a = lead * (l > 0)
    b = np.sqrt(np.where(inside, (l + 1) ** 2 - rows[:, None] ** 2, 0) / (4.0 * (l + 1) ** 2 - 1))
    b[:, -1] = 0
    self.gradient = tensor((l + 1) * a), tensor(-l * b)
    self.divergence = tensor((l - 1) * a), tensor(-(l + 2) * b)
    self.eigenvalues = tensor(-l * (l + 1.0))
    self.inverse_eigenvalues = tensor(np.where(l > 0, -1.0 / np.maximum(l * (l + 1.0), 1), 0.0))
    self.rows = tensor(rows)
    self.clip = tensor((l < L - 1) * 1.0)

  def to_nodal(self, x):
    lead = x.shape[:-2]
    x = x.reshape(-1, 2 * self.M - 1, self.L)
    x = torch.cat([x[:, :1], torch.zeros_like(x[:, :1]), x[:, 1:]], 1)
    B = x.shape[0]
    x = x.reshape(B, self.M, 2, self.L).permute(1, 2, 0, 3).reshape(self.M, 2 * B, self.L)
    rows = torch.bmm(x, self.P.transpose(1, 2).contiguous())
    z = self.F @ rows.reshape(2 * self.M, B * self.J)
    return z.reshape(self.I, B, self.J).permute(1, 0, 2).reshape(lead + (self.I, self.J))

  def to_modal(self, z):
    lead = z.shape[:-2]
    z = (z * self.weights).reshape(-1, self.I, self.J)
    B = z.shape[0]
    rows = self.F.T.contiguous() @ z.permute(1, 0, 2).reshape(self.I, B * self.J)
    x = torch.bmm(rows.reshape(self.M, 2 * B, self.J), self.P)
    x = x.reshape(self.M, 2, B, self.L).permute(2, 0, 1, 3).reshape(B, 2 * self.M, self.L)
    return torch.cat([x[:, :1], x[:, 2:]], 1).reshape(lead + (2 * self.M - 1, self.L))

  def d_dlon(self, x):
    cos, sin = x[..., 1::2, :], x[..., 2::2, :]
    m = self.rows[1::2, None]
    pairs = torch.stack([m * sin, -m * cos], -2)
    return torch.cat([torch.zeros_like(x[..., :1, :]), pairs.flatten(-3, -2)], -2)

  def _two_point(self, weights, x):
    up, down = weights
    zero = torch.zeros_like(x[..., :1])
    return torch.cat([(up * x)[..., 1:], zero], -1) + torch.cat([zero, (down * x)[..., :-1]], -1)

  def d_dlat(self, x):  # cos(lat) d/dlat
    return self._two_point(self.gradient, x)

  def d_dlat_cos2(self, x):  # sec(lat) d/dlat cos(lat)^2
    return self._two_point(self.divergence, x)

  def div(self, u, v):
    return self.d_dlon(u) + self.d_dlat_cos2(v)

  def curl(self, u, v):
    return self.d_dlon(v) - self.d_dlat_cos2(u)

  def cos_winds(self, z, d):
    psi, chi = z * self.inverse_eigenvalues, d * self.inverse_eigenvalues
    return self.d_dlon(chi) - self.d_dlat(psi), self.d_dlat(chi) + self.d_dlon(psi)


class _Equations:
  """Sigma-level primitive equations on one member's leaves, float64."""

  def __init__(self, case, seed):
    self.case = case
    self.sphere = _Sphere(case['grid'])
    self.orography = _orography(case['grid'], seed).to(_dtype(case)).double()
    self.specs = units_lib.SimUnits.from_si()
    K = case['layers']
    vertical = sigma_coordinates.SigmaCoordinates.equidistant(K)
    tensor = lambda a: torch.as_tensor(np.asarray(a, np.float64), device=DEVICE)  # noqa: E731
    column = lambda a: tensor(a)[:, None, None]  # noqa: E731
    # the levels are float32 numbers, and so are the constants made from them
    alpha = np.diff(np.log(vertical.centers), append=0) / 2
    alpha[-1] = -np.log(vertical.centers[-1])
    thickness = vertical.layer_thickness
    pair = np.concatenate([[0.0], alpha[1:] + alpha[:-1]])
    upper = np.triu(np.ones((K, K)), 1) * pair + np.diag(alpha)
    lower = np.tril(np.ones((K, K)))
    pressure = lower * alpha[:, None]
    above = np.concatenate([np.zeros((1, K)), pressure[:-1]])
    scale = self.specs.kappa * REFERENCE_TEMPERATURE
    self.G = self.specs.R * tensor(upper)
    self.H = tensor(scale * (pressure + above) / thickness[:, None] * thickness)
    self.alpha, self.thickness = column(alpha), column(thickness)
    self.sigma = column(vertical.centers)
    self.depth = column(np.maximum(0, (vertical.centers - 0.7) / (1 - 0.7)))
    self.sums = column(np.cumsum(thickness)[:-1])
    self.inverse_spacing = column(1 / vertical.center_to_center)
    self.inverses = {}

  def advection(self, flux, x):
    w = flux * torch.diff(x, dim=0) * self.inverse_spacing
    zero = torch.zeros_like(x[:1])
    return -0.5 * (torch.cat([w, zero]) + torch.cat([zero, w]))

  def explicit(self, x):
    s, p, moist = self.sphere, self.specs, self.case['moist']
    names = TRACERS if moist else ()
    uc, vc = s.cos_winds(x['vorticity'], x['divergence'])
    lnps = x['log_surface_pressure']
    modal = [x['vorticity'], x['divergence'], x['temperature_variation'], uc, vc, s.d_dlon(lnps),
             s.d_dlat(lnps)] + [x[k] for k in names]
    if moist:
      q = x[TRACERS[0]]
      modal += [lnps * s.eigenvalues, s.d_dlon(q), s.d_dlat(q)]
    parts = torch.split(s.to_nodal(torch.cat(modal)), [len(f) for f in modal])
    zeta, delta, temp, u, v, px, py = parts[:7]
    tracers = dict(zip(names, parts[7:]))
    sec2 = 1 / s.cos2
    absolute = zeta + 2 * p.angular_velocity * s.sin_lat
    advected = (u * px + v * py) * sec2
    total = torch.cumsum((delta + advected) * self.thickness, 0)
    partial = torch.cumsum(advected * self.thickness, 0)
    flux = self.sums * total[-1:] - total[:-1]
    tref = REFERENCE_TEMPERATURE
    virtual, thermal, thermal_ref = 1.0, temp, 0.0
    if moist:
      humid = tracers[TRACERS[0]]
      ratio, heat = p.R_vapor / p.R, p.Cp_vapor / p.Cp
      virtual = 1 + (ratio - 1) * humid - tracers[TRACERS[1]] - tracers[TRACERS[2]]
      thermal = temp * (1 + (ratio - 1) * humid) / (1 + (heat - 1) * humid)
      thermal_ref = tref * (ratio - heat) * humid / (1 + (heat - 1) * humid)

    def omega(field, prefix):
      weighted = self.alpha * prefix
      shifted = torch.cat([torch.zeros_like(weighted[:1]), weighted[:-1]])
      return field * (advected - (weighted + shifted) / self.thickness)

    rt = p.R * temp * virtual
    fu = (-v * absolute - self.advection(flux, u) + rt * px) * sec2
    fv = (u * absolute - self.advection(flux, v) + rt * py) * sec2
    heating = (temp * delta + self.advection(flux, temp)
               + p.kappa * (omega(tref, partial) + omega(thermal + thermal_ref, total)))
    energy = (u * u + v * v) * sec2 / 2
    nodal = [fu, fv, energy, heating, u * temp * sec2, v * temp * sec2, -partial[-1:]]
    for k in names:
      t = tracers[k]
      nodal += [self.advection(flux, t) + t * delta, u * t * sec2, v * t * sec2]
    if moist:
      lap, qx, qy = parts[7 + len(names):]
      excess = tref * (p.R_vapor - p.R)
      warm = humid * (temp + tref) * (p.R_vapor / p.R - 1)
      nodal += [excess * sec2 * (px * qy - py * qx), torch.einsum('gh,hij->gij', self.G, warm),
                excess * (sec2 * (qx * px + qy * py) + humid * lap)]
    parts = torch.split(s.to_modal(torch.cat(nodal)), [len(f) for f in nodal])
    fu, fv, energy, heating, tu, tv, pressure = parts[:7]
    lap = s.eigenvalues
    out = {'vorticity': -s.curl(fu, fv),
           'divergence': -s.div(fu, fv) - lap * (energy + p.g * self.orography),
           'temperature_variation': heating - s.div(tu, tv),
           'log_surface_pressure': pressure}
    for i, k in enumerate(names):
      t, tu, tv = parts[7 + 3 * i:10 + 3 * i]
      out[k] = t - s.div(tu, tv)
    if moist:
      curl, geo, dot = parts[7 + 3 * len(names):]
      out['vorticity'] = out['vorticity'] + curl
      out['divergence'] = out['divergence'] - lap * geo - dot
    out = {k: t * s.clip for k, t in out.items()}
    if self.case.get('held_suarez'):
      for k, t in self.relaxation(x).items():
        out[k] = out[k] + t
    return out

  def relaxation(self, x):
    """Held-Suarez drag and relaxation with the default parameters."""
    s, p = self.sphere, self.specs
    day = p.nondimensionalize(1.0 * units_lib.scales.units.day)
    uc, vc = s.cos_winds(x['vorticity'], x['divergence'])
    u, v, temp, lnps = (s.to_nodal(t) for t in (uc, vc, x['temperature_variation'],
                                                 x['log_surface_pressure']))
    ratio = self.sigma * torch.exp(lnps) / _p0()
    equilibrium = torch.clamp(
        ratio ** p.kappa * (315 - 60 * s.sin_lat ** 2 - 10 * torch.log(ratio) * s.cos2), min=200)
    slow, fast = 1 / (40 * day), 1 / (4 * day)
    rate = slow + (fast - slow) * self.depth * s.cos2 ** 2
    drag = self.depth / day / s.cos2
    fu, fv = s.to_modal(-drag * u), s.to_modal(-drag * v)
    cooling = s.to_modal(-rate * (REFERENCE_TEMPERATURE + temp - equilibrium))
    return {'vorticity': s.curl(fu, fv) * s.clip, 'divergence': s.div(fu, fv) * s.clip,
            'temperature_variation': cooling}

  def levels(self, matrix, x):
    return torch.einsum('gh,hml->gml', matrix, x)

  def implicit(self, x):
    lap = self.sphere.eigenvalues
    d, t, q = (x[k] for k in FIELDS[1:])
    rt = self.specs.R * REFERENCE_TEMPERATURE
    return {'divergence': -lap * (self.levels(self.G, t) + rt * q),
            'temperature_variation': -self.levels(self.H, d),
            'log_surface_pressure': -(self.thickness * d).sum(0, keepdim=True)}

  def solve(self, x, eta):
    """(1 - eta implicit)^-1, one dense matrix per degree."""
    K = self.case['layers']
    if eta not in self.inverses:
      lap = self.sphere.eigenvalues[:, None, None]
      a = torch.eye(2 * K + 1, dtype=torch.float64, device=DEVICE).repeat(len(lap), 1, 1)
      a[:, :K, K:2 * K] = eta * lap * self.G
      a[:, :K, 2 * K] = eta * lap[:, 0] * self.specs.R * REFERENCE_TEMPERATURE
      a[:, K:2 * K, :K] = eta * self.H
      a[:, 2 * K, :K] = eta * self.thickness[:, 0, 0]
      self.inverses[eta] = torch.as_tensor(np.linalg.inv(a.cpu().numpy()), device=DEVICE)
    columns = torch.cat([x[k] for k in FIELDS[1:]]).permute(2, 0, 1).contiguous()
    d, t, q = torch.split(torch.bmm(self.inverses[eta], columns).permute(1, 2, 0), [K, K, 1])
    return {**x, 'divergence': d, 'temperature_variation': t, 'log_surface_pressure': q}

  def step(self, x, dt):
    """SIL3 (Whitaker and Kar 2013) and the exponential filter."""
    a_ex = [[1 / 3], [1 / 6, 1 / 2], [1 / 2, -1 / 2, 1]]
    a_im = [[1 / 6, 1 / 6], [1 / 3, 0, 1 / 3], [3 / 8, 0, 3 / 8, 1 / 4]]
    f, g = [self.explicit(x)], [self.implicit(x)]

    def combine(ex, im):
      out = {}
      for k in x:
        out[k] = x[k] + dt * sum(c * t[k] for c, t in zip(ex, f) if c)
        if k in g[0]:
          out[k] = out[k] + dt * sum(c * t[k] for c, t in zip(im, g) if c)
      return out

    for i in range(3):
      y = self.solve(combine(a_ex[i], a_im[i][:-1]), dt * a_im[i][-1])
      if i < 2:
        f.append(self.explicit(y))
      g.append(self.implicit(y))
    l = torch.arange(self.sphere.L, device=DEVICE, dtype=torch.float64)
    scaling = torch.exp(-dt / 0.010938 * (l / l[-1]) ** 36)
    return {k: t * scaling for k, t in combine([1 / 2, -1 / 2, 1], [3 / 8, 0, 3 / 8, 1 / 4]).items()}


def _exact_transform(case, seed):
  s = _Sphere(case['grid'])
  x = [t.double() for t in _transform_inputs(case, seed)]
  nodal = s.to_nodal(x[0])
  out = [nodal, s.to_modal(nodal)]
  if case['gradient']:
    # adjoints: to_nodal^T is to_modal without the quadrature weights, and back
    nodal_cotangent = x[1] + s.to_nodal(x[2]) * s.weights
    out.append(s.to_modal(nodal_cotangent / s.weights))
  return out


def _exact_winds(case, seed):
  s = _Sphere(case['grid'])
  z, d = (t.double() for t in _wind_inputs(case, seed))
  u, v = (s.to_nodal(t * s.clip) / torch.sqrt(s.cos2) for t in s.cos_winds(z, d))
  mu, mv = (s.to_modal(t / torch.sqrt(s.cos2)) for t in (u, v))
  return [u, v, s.curl(mu, mv) * s.clip, s.div(mu, mv) * s.clip]


def _exact_member(case, equations, leaves, targets):
  """Outputs of one member; the loss is this member's share of the mean."""
  if case['kind'] == 'explicit':
    return equations.explicit(leaves)
  dt = _time_step(case)
  if case['kind'] == 'step':
    for _ in range(case['steps']):
      leaves = equations.step(leaves, dt)
    return leaves
  leaves = {k: t.requires_grad_(True) for k, t in leaves.items()}
  final = leaves
  for _ in range(case['steps']):
    final = equations.step(final, dt)
  loss = _loss(equations.sphere.to_nodal, final, targets, case['layers']) / case['members']
  names = _names(case)
  gradients = torch.autograd.grad(loss, [leaves[k] for k in names])
  return dict(loss=loss.detach(), state={k: final[k].detach() for k in names},
              gradients=dict(zip(names, gradients)))


def exact(case, seed):
  if case['kind'] == 'transform':
    return _exact_transform(case, seed)
  if case['kind'] == 'winds':
    return _exact_winds(case, seed)
  equations = _Equations(case, seed)
  leaves = {k: t.to(_dtype(case)).double() for k, t in _state_arrays(case, seed).items()}
  lead = leaves['vorticity'].shape[:-3]
  targets = None
  if case['kind'] == 'adjoint':
    _, _, I, J = _shape(case['grid'])
    targets = [t.to(_dtype(case)).double() for t in _targets(case, seed, lead + (I, J))]
  if not lead:
    return _exact_member(case, equations, leaves, targets)
  members = []
  for e in range(case['members']):
    member_targets = [t[e] for t in targets] if targets else None
    members.append(_exact_member(case, equations, {k: t[e].clone() for k, t in leaves.items()},
                                 member_targets))
  stack = lambda key: {k: torch.stack([m[key][k] for m in members])  # noqa: E731
                       for k in members[0][key]}
  if case['kind'] != 'adjoint':
    return {k: torch.stack([m[k] for m in members]) for k in _names(case)}
  return dict(loss=sum(m['loss'] for m in members), state=stack('state'),
              gradients=stack('gradients'))
