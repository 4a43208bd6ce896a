"""Nodal kernel with a column's levels split over the waves of a block (small
batches) and with whole columns (large ones) against the unfused formulation."""
import numpy as np
import pytest
import torch

from dinosaur_amd import coordinate_systems, primitive_equations as pe
from dinosaur_amd import sigma_coordinates, spherical_harmonic as sh, units

pytestmark = pytest.mark.gpu

FIELDS = ('vorticity', 'divergence', 'temperature_variation', 'log_surface_pressure')
CLOUDS = ('cloud_a', 'cloud_b')


def _ragged():
  # 200 columns: three blocks of 64 and one of 8
  return sh.Grid(longitude_wavenumbers=7, total_wavenumbers=8, longitude_nodes=20,
                 latitude_nodes=10)


# Levels: one wave (1 to 3), an uneven share (5, 17, 37), the model's (12);
# 4 and 5 members of T42 L8 lie on both sides of the batches where the whole-column
# kernel takes over, 12 and 13 members of two levels both beyond.
@pytest.mark.parametrize('grid,K,members,moist,tref_varies', [
    (_ragged, 1, 1, False, False), (_ragged, 2, 3, True, True), (_ragged, 3, 1, False, True),
    (_ragged, 5, 2, True, False), (_ragged, 17, 1, True, True), (_ragged, 37, 2, False, True),
    (sh.Grid.T21, 12, 1, True, True), (sh.Grid.T42, 2, 12, True, True),
    (sh.Grid.T42, 2, 13, True, True), (sh.Grid.T42, 8, 4, True, True),
    (sh.Grid.T42, 8, 5, True, True)])
def test_split_and_whole_columns_match_unfused(grid, K, members, moist, tref_varies, gpu_device):
  grid = grid()
  coords = coordinate_systems.CoordinateSystem(
      grid, sigma_coordinates.SigmaCoordinates.equidistant(K))
  names = ['specific_humidity', *CLOUDS] if moist else ['passive']
  kw = dict(humidity_key='specific_humidity', cloud_keys=CLOUDS) if moist else {}
  tref = np.linspace(220., 290., K) if tref_varies else np.full(K, 250.0)
  rs = np.random.RandomState(K + members)
  l = grid.modal_mesh[1]

  def field(lead, amp):
    x = rs.normal(size=(members, lead) + grid.modal_shape) * grid.mask * amp / (l + 1) ** 1.5
    return torch.as_tensor(x, device=gpu_device)

  lnps = field(1, 0.05)
  lnps[..., 0, 0] += 3.5449077 * 4.0
  st = pe.State(field(K, 0.1), field(K, 0.1), field(K, 5.0), lnps,
                tracers={n: field(K, 1e-3) for n in names})
  oro = torch.as_tensor(rs.normal(size=grid.modal_shape) * grid.mask * 1e-4, device=gpu_device)
  a, b = (pe.PrimitiveEquationsSigma(tref, oro, coords, units.SimUnits.from_si(),
                                     fused_nodal=fused, **kw).explicit_terms(st)
          for fused in (True, False))
  pairs = [(f, getattr(a, f), getattr(b, f)) for f in FIELDS]
  pairs += [(n, a.tracers[n], b.tracers[n]) for n in names]
  for name, x, y in pairs:
    # Only the order of sums differs: a few K eps = 1e-14 of the largest terms, which
    # the divergence's Laplacian leaves up to 1e2 times larger than their sum.
    err = (x - y).abs().max().item() / max(y.abs().max().item(), 1e-300)
    assert err < 1e-12, (name, err)


# 200 columns a member: 600 members lie beyond the split form's batches, one within
# (from 4 levels on).
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('K,moist,tref_varies', [(1, False, False), (2, True, True),
                                                 (3, False, True), (5, True, False),
                                                 (8, False, True), (17, True, True),
                                                 (37, True, True), (64, True, False)])
def test_member_in_a_batch_equals_the_member_alone(gpu_device, K, moist, tref_varies, dtype):
  print('[test] nodal member alone', K, moist, dtype, flush=True)
  members = 600
  coords = coordinate_systems.CoordinateSystem(
      _ragged(), sigma_coordinates.SigmaCoordinates.equidistant(K))
  names = ['specific_humidity', *CLOUDS] if moist else ['passive']
  kw = dict(humidity_key='specific_humidity', cloud_keys=CLOUDS) if moist else {}
  tref = np.linspace(220., 290., K) if tref_varies else np.full(K, 250.0)
  eq = pe.PrimitiveEquationsSigma(tref, np.zeros(coords.horizontal.modal_shape), coords,
                                  units.SimUnits.from_si(), **kw)
  handle = eq._nodal_handle(gpu_device, names)
  # levels of the input groups: Z D T, tracers, U V, GX GY, moist LP QX QY
  levels = [K] * (5 + len(names)) + [1, 1] + ([1, K, K] if moist else [])
  gen = torch.Generator(device=gpu_device).manual_seed(K)
  groups = [torch.randn((members, n) + coords.horizontal.nodal_shape, generator=gen, dtype=dtype,
                        device=gpu_device) for n in levels]

  def run(first, last):
    x = torch.cat([g[first:last].flatten(0, 1) for g in groups])
    out = pe._NodalFused.apply(x, handle, last - first)
    # CU CV KE TEMP UT VT, LSP, three a tracer, moist CURL DC
    n_out = [K] * 6 + [1] + [K] * (3 * len(names) + (2 if moist else 0))
    return [f.unflatten(0, (last - first, n))
            for n, f in zip(n_out, out.split([n * (last - first) for n in n_out]))]

  whole = run(0, members)
  for e in (0, 1, members - 1):
    assert all(x[e:e + 1].equal(y) for x, y in zip(whole, run(e, e + 1)))
