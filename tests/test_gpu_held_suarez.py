"""Held-Suarez forcing fused into the primitive equations' explicit terms
against the sum of the two equations' own explicit terms, values and
gradients, at level counts around the kernel's four-way split; and IMEX steps
of the composed equation against the stage-by-stage path.

Tolerances, normwise: the fused terms add the drag and relaxation before the
forward transform instead of after it, so the two differ by the rounding of
the transforms (u sqrt(I), see test_gpu_dft.py, times the cancellation of the
divergence tendency's large terms, about 1e2): 1e-12 in FP64; 2e-4 in FP32.
"""
import numpy as np
import pytest
import torch

from dinosaur_amd import _lib, held_suarez, primitive_equations as pe, time_integration as ti
from dinosaur_amd import units, workloads

pytestmark = pytest.mark.gpu

TOL = {torch.float64: 1e-12, torch.float32: 2e-4}


def _setup(K, members, moist, dtype, dev, name='T21'):
  eq, st, coords, ps = workloads.build_primitive(name, K, members=members, moist=moist,
                                                 dtype=dtype, device=dev)
  gen = torch.Generator(device=dev).manual_seed(K)
  mask = torch.as_tensor(coords.horizontal.mask, device=dev)
  bump = lambda x, a: x + a * mask * torch.randn(x.shape, generator=gen, device=dev, dtype=dtype)  # noqa: E731
  st = pe.State(bump(st.vorticity, 1e-2), bump(st.divergence, 1e-3),
                bump(st.temperature_variation, 2.0), bump(st.log_surface_pressure, 1e-3),
                st.tracers)
  hs = held_suarez.HeldSuarezForcingSigma(coords, ps, eq.reference_temperature)
  return eq, hs, st, coords, ps


def _leaves(st):
  return [getattr(st, f) for f in st._ARRAYS] + list(st.tracers.values())


def _close(a, b, tol, what):
  for i, (x, y) in enumerate(zip(_leaves(a), _leaves(b))):
    d = (x.double() - y.double()).norm() / y.double().norm().clamp(min=1e-300)
    assert d <= tol or x.equal(y), (what, i, d.item())


@pytest.mark.parametrize('dtype', [torch.float64, torch.float32])
@pytest.mark.parametrize('K,members,moist', [(1, 1, False), (3, 2, False), (5, 1, True),
                                             (8, 1, False), (13, 3, True)])
def test_fused_terms_equal_the_sum(gpu_device, K, members, moist, dtype):
  print('[test] held-suarez fused', K, members, moist, dtype, flush=True)
  eq, hs, st, *_ = _setup(K, members, moist, dtype, gpu_device)
  forced = hs.fused_with(eq)
  assert forced is not None
  names = list(st.tracers)

  def run(fn):
    xs = [x.clone().requires_grad_(True) for x in _leaves(st)]
    out = fn(pe.State(*xs[:4], dict(zip(names, xs[4:]))))
    gen = torch.Generator(device=gpu_device).manual_seed(1)
    cot = [torch.randn(x.shape, generator=gen, device=gpu_device, dtype=dtype)
           for x in _leaves(out)]
    grads = torch.autograd.grad(_leaves(out), xs, cot, allow_unused=True)
    grads = [torch.zeros_like(x) if g is None else g for g, x in zip(grads, xs)]
    return out, pe.State(*grads[:4], dict(zip(names, grads[4:])))

  got, ggot = run(forced.explicit_terms)
  ref, gref = run(lambda s: ti._tree_sum([eq.explicit_terms(s), hs.explicit_terms(s)]))
  mask = torch.as_tensor(eq.coords.horizontal.mask, device=gpu_device)
  tri = lambda s: s.tree_map_arrays(lambda x: x * mask)  # noqa: E731
  _close(got, ref, TOL[dtype], 'value')
  _close(tri(ggot), tri(gref), TOL[dtype], 'gradient')


def test_composed_step_uses_the_fused_path(gpu_device):
  eq, hs, st, coords, ps = _setup(6, 2, False, torch.float64, gpu_device)
  dt = ps.nondimensionalize(600.0 * units.scales.units.s)
  composed = ti.compose_equations([hs, eq])
  assert composed._flat_imex_ops(st.as_flat()) is not None
  plain = ti.compose_equations([eq, hs])
  plain._flat_imex_ops = lambda state: None
  filters = [ti.exponential_step_filter(coords.horizontal, dt)]
  a, b = (ti.step_with_filters(ti.imex_rk_sil3(e, dt), filters) for e in (composed, plain))
  st.sim_time = 1.5
  x, y = a(a(st)), b(b(st))
  assert x.sim_time == y.sim_time
  _close(x, y, 1e-12, 'step')


def test_pairs_the_kernels_do_not_serve_stay_unfused(gpu_device):
  eq, hs, *_ = _setup(4, 1, False, torch.float64, gpu_device)
  other, *_ = _setup(5, 1, False, torch.float64, gpu_device)
  assert hs.fused_with(other) is None
  eq.fused_nodal = False
  assert hs.fused_with(eq) is None

  class Mine(pe.PrimitiveEquationsSigma):
    def explicit_terms(self, state):
      return super().explicit_terms(state)

  eq.fused_nodal = True
  mine = Mine(eq.reference_temperature, eq.orography, eq.coords, eq.physics_specs)
  assert hs.fused_with(mine) is None


@pytest.mark.parametrize('name', ['kf', 'ka', 'ks', 'sigma_b', 'sigma', 'reference_temperature',
                                  'lat', 'minT', 'p0'])
def test_changed_parameters_are_used(gpu_device, name):
  """After a parameter changes, a forcing that has run equals a new one, fused
  and by itself."""
  eq, hs, st, coords, ps = _setup(6, 1, False, torch.float64, gpu_device)
  run = lambda forcing: (forcing.fused_with(eq).explicit_terms(st), forcing.explicit_terms(st))  # noqa: E731
  before = run(hs)
  new = held_suarez.HeldSuarezForcingSigma(coords, ps, eq.reference_temperature)
  for forcing in (hs, new):
    setattr(forcing, name, getattr(forcing, name) * 0.9)
  for b, x, y in zip(before, run(hs), run(new)):
    assert all(p.equal(q) for p, q in zip(_leaves(x), _leaves(y)))
    assert not all(p.equal(q) for p, q in zip(_leaves(b), _leaves(x)))


def test_work_of_the_forcing_kernels(gpu_device):
  """Fields that the kernels read and write (8 K + 1 forward, 9 K + 2 adjoint)."""
  K, members = 5, 2
  eq, hs, st, coords, _ = _setup(K, members, False, torch.float32, gpu_device)
  x = st.as_flat().flat_buffer().clone().requires_grad_(True)
  state = pe.State.from_flat(x, (members,), K, ())
  field = 4 * coords.horizontal.nodal_shape[0] * coords.horizontal.nodal_shape[1]
  with _lib.work_tally() as t:
    out = hs.fused_with(eq).explicit_terms(state).flat_buffer()
    forward = t.families['held_suarez']['bytes']
    out.sum().backward()
  assert forward == field * members * (8 * K + 1)
  assert t.families['held_suarez']['bytes'] - forward == field * members * (9 * K + 2)
