"""compose_equations of the primitive equations and the Held-Suarez forcing:
the fused step serves only the two classes' own methods, and the arguments of
its one-call form hold what they point to (host side)."""
import copy
import gc
import weakref

import numpy as np
import pytest
import torch

from dinosaur_amd import coordinate_systems, held_suarez, primitive_equations as pe
from dinosaur_amd import sigma_coordinates, spherical_harmonic as sh, time_integration as ti, units


def _pair(K=4):
  coords = coordinate_systems.CoordinateSystem(
      sh.Grid(8, 9, 24, 12), sigma_coordinates.SigmaCoordinates.equidistant(K))
  ps = units.SimUnits.from_si()
  tref = np.full(K, 288.0)
  eq = pe.PrimitiveEquationsSigma(tref, np.zeros(coords.horizontal.modal_shape), coords, ps)
  return eq, held_suarez.HeldSuarezForcingSigma(coords, ps, tref)


@pytest.mark.parametrize('name', ['explicit_terms', '_explicit_fused', 'implicit_terms',
                                  'implicit_inverse'])
def test_methods_replaced_on_the_equation_stay_unfused(name):
  eq, hs = _pair()
  assert hs.fused_with(eq) is not None
  setattr(eq, name, getattr(eq, name))
  assert hs.fused_with(eq) is None


@pytest.mark.parametrize('name', ['explicit_terms', 'equilibrium_temperature', 'kv', 'kt'])
def test_methods_replaced_on_the_forcing_stay_unfused(name):
  eq, hs = _pair()
  setattr(hs, name, getattr(hs, name))
  assert hs.fused_with(eq) is None


@pytest.mark.parametrize('name', ['explicit_terms', 'implicit_terms', 'implicit_inverse'])
def test_methods_replaced_on_the_composed_equation_are_used(name, monkeypatch):
  class Flat:
    def as_flat(self):
      return self

  def replaced(*args):
    raise NotImplementedError

  monkeypatch.setattr(held_suarez._ForcedEquations, 'flat_imex_ops', lambda self, state: 'ops')
  monkeypatch.setattr(ti, '_fused_imex_step', lambda *args: 'fused')
  eq, hs = _pair()
  monkeypatch.setattr(pe.PrimitiveEquationsSigma, 'implicit_inverse', lambda *args: 0.0)
  composed = ti.compose_equations([eq, hs])
  assert ti.imex_rk_sil3(composed, 0.1)(Flat()) == 'fused'
  mine = copy.copy(composed)
  setattr(mine, name, replaced)
  for other in {'explicit_terms', 'implicit_terms'} - {name}:
    setattr(mine, other, lambda state: 0.0)
  monkeypatch.setattr(ti, '_stage', lambda *args: 0.0)
  with pytest.raises(NotImplementedError):
    ti.imex_rk_sil3(mine, 0.1)(Flat())
  assert ti.imex_rk_sil3(composed, 0.1)(Flat()) == 'fused'


def test_explicit_fused_replaced_on_the_equation_is_not_one_call():
  eq, _ = _pair()
  eq._explicit_fused = lambda *args: None
  assert eq._native_args(torch.zeros(13, 15, 9), 1, []) is None


def test_one_call_arguments_hold_what_they_point_to(monkeypatch):
  """A handle that another thread drops from the caches stays alive with them."""
  class Handle:
    handle, tuned = 1, None

  eq, hs = _pair()
  monkeypatch.setattr(sh.RealSphericalHarmonics, 'plan', lambda self, device: Handle())
  made = []

  def make(*args):
    h = Handle()
    made.append(weakref.ref(h))
    return h

  eq._modal_handle = eq._nodal_handle = hs.handle = make
  args = eq._native_args(torch.zeros(13, 15, 9), 1, [], hs)
  eq._consts.clear()
  gc.collect()
  assert len(made) == 3 and all(r() is not None for r in made)
  assert any(isinstance(t, torch.Tensor) and t.data_ptr() == args.orography for t in args.owners)


@pytest.mark.parametrize('name', ['explicit_terms', '_explicit_fused'])
def test_replaced_explicit_terms_get_whole_stage_values(name):
  """Stage values may leave the entries below the triangle unwritten only for the
  kernels that skip them."""
  eq, _ = _pair()
  assert pe._FlatImexOps(eq, ((), 4, ()), 1).stage_triangle_only
  setattr(eq, name, getattr(eq, name))
  assert not pe._FlatImexOps(eq, ((), 4, ()), 1).stage_triangle_only
