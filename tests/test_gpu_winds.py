"""Fused wind conversions (vor_div_to_uv_nodal, uv_nodal_to_vor_div_modal)
against the composed grid operators in FP64, values and gradients, over grids
with and without a clipped top degree, latitude spacings, leading shapes,
strides and entries below the triangle.

Tolerance, normwise: 1e-12 in FP64 (1e-9 on the equiangular grid, whose
quadrature weights and 1 / cos(lat) span nine decades), 2e-3 in FP32 for the
divergence, a small difference of large terms (2e-5 for the winds).
"""
import functools

import numpy as np
import pytest
import torch

from dinosaur_amd import spherical_harmonic as sh

pytestmark = pytest.mark.gpu


def _composed_uv(grid, z, d, clip):
  u, v = sh.get_cos_lat_vector(z, d, grid, clip=clip)
  cos = grid.const('cos_lat', z.device, z.dtype)
  return grid.to_nodal(u) / cos, grid.to_nodal(v) / cos


def _composed_vor_div(grid, u, v, clip):
  cos = grid.const('cos_lat', u.device, u.dtype)
  uc, vc = grid.to_modal(u / cos), grid.to_modal(v / cos)
  return grid.curl_cos_lat((uc, vc), clip=clip), grid.div_cos_lat((uc, vc), clip=clip)


def _rel(a, b):
  return ((a.double() - b.double()).norm() / b.double().norm()).item()


GRIDS = [sh.Grid.T21(), sh.Grid.TL31(), sh.Grid.with_wavenumbers(22, radius=2.5),
         sh.Grid.with_wavenumbers(43, dealiasing='linear'),
         sh.Grid(16, 17, 48, 25, 'equiangular'), sh.Grid.T106()]


@pytest.mark.parametrize('dtype', [torch.float64, torch.float32])
@pytest.mark.parametrize('clip', [True, False])
@pytest.mark.parametrize('index', range(len(GRIDS)))
def test_winds_match_composed_operators(gpu_device, index, clip, dtype):
  grid = GRIDS[index]
  print('[test] winds', grid.nodal_shape, clip, dtype, flush=True)
  gen = torch.Generator(device=gpu_device).manual_seed(index)
  tol = 1e-9 if grid.latitude_spacing != 'gauss' else 1e-12
  tol, dtol = (tol, tol) if dtype == torch.float64 else (2e-5, 2e-3)
  mask = torch.as_tensor(grid.mask, device=gpu_device)
  l = torch.arange(grid.modal_shape[1], device=gpu_device) + 1.0
  for lead in ((), (3,), (2, 5)):
    z, d = (torch.randn(lead + grid.modal_shape, generator=gen, device=gpu_device,
                        dtype=torch.float64) / l for _ in range(2))
    z, d = z.to(dtype), (0.1 * d).to(dtype)  # entries below the triangle included
    if lead:  # not contiguous
      z = z.transpose(-1, -2).contiguous().transpose(-1, -2)
    z, d = z.requires_grad_(True), d.requires_grad_(True)
    z64, d64 = (t.detach().double().requires_grad_(True) for t in (z, d))
    got = sh.vor_div_to_uv_nodal(grid, z, d, clip=clip)
    ref = _composed_uv(grid, z64, d64, clip)
    assert max(_rel(a, b) for a, b in zip(got, ref)) <= tol
    cot = [torch.randn(t.shape, generator=gen, device=gpu_device, dtype=torch.float64)
           for t in ref]
    ggot = torch.autograd.grad(got, (z, d), [c.to(dtype) for c in cot])
    gref = torch.autograd.grad(ref, (z64, d64), cot)
    assert max(_rel(a * mask, b * mask) for a, b in zip(ggot, gref)) <= max(tol, 2e-12)

    u, v = (t.detach().clone().requires_grad_(True) for t in got)
    u64, v64 = (t.detach().double().requires_grad_(True) for t in (u, v))
    got = sh.uv_nodal_to_vor_div_modal(grid, u, v, clip=clip)
    ref = _composed_vor_div(grid, u64, v64, clip)
    assert max(_rel(a, b) for a, b in zip(got, ref)) <= dtol
    assert all((t.detach()[..., ~mask] == 0).all() for t in got)
    cot = [torch.randn(t.shape, generator=gen, device=gpu_device, dtype=torch.float64) * mask
           for t in ref]
    ggot = torch.autograd.grad(got, (u, v), [c.to(dtype) for c in cot])
    gref = torch.autograd.grad(ref, (u64, v64), cot)
    assert max(_rel(a, b) for a, b in zip(ggot, gref)) <= max(tol, 2e-12)


def test_winds_outputs_are_independent(gpu_device):
  grid = GRIDS[0]
  z = torch.randn((2,) + grid.modal_shape, device=gpu_device)
  u, v = sh.vor_div_to_uv_nodal(grid, z, z)
  before = v.clone()
  u.mul_(2.0)
  assert v.equal(before) and u.is_contiguous() and v.is_contiguous()
  x = z.clone().requires_grad_(True)
  u, v = sh.vor_div_to_uv_nodal(grid, x, x)
  w = (v * v).sum()
  u.mul_(2.0)  # v, saved for the product's backward, is not u's memory
  torch.autograd.grad(w + u.sum(), x)
  out = sh.vor_div_to_uv_nodal(grid, z.cpu().numpy(), z.cpu().numpy())
  assert all(isinstance(a, np.ndarray) for a in out)


def test_one_degree_takes_the_composed_operators(gpu_device):
  grid = sh.Grid(1, 1, 4, 2)
  z, d = (torch.randn((3, 1, 1), device=gpu_device) for _ in range(2))
  for a, b in zip(sh.vor_div_to_uv_nodal(grid, z, d), _composed_uv(grid, z, d, True)):
    assert a.shape == (3, 4, 2) and a.equal(b)
  u, v = (torch.randn((3, 4, 2), device=gpu_device) for _ in range(2))
  for a, b in zip(sh.uv_nodal_to_vor_div_modal(grid, u, v, clip=False),
                  _composed_vor_div(grid, u, v, False)):
    assert a.shape == (3, 1, 1) and a.equal(b)


def test_changing_one_output_leaves_the_other_usable_by_autograd(gpu_device):
  grid = GRIDS[0]
  z = torch.randn((2,) + grid.modal_shape, device=gpu_device)
  w = torch.randn((2,) + grid.nodal_shape, device=gpu_device)
  for a, b in (sh.vor_div_to_uv_nodal(grid, z, z), sh.uv_nodal_to_vor_div_modal(grid, w, w)):
    a.requires_grad_()
    y = (a * a).sum()
    b.mul_(2.0)
    y.backward()
    assert a.grad.equal(2 * a.detach())


def test_equal_grids_share_one_handle(gpu_device):
  """Also grids made with a functools.partial of their own, which compare unequal."""
  def handle(**kw):
    impl = functools.partial(sh.RealSphericalHarmonics, transform_precision='float32')
    grid = sh.Grid(8, 9, 24, 12, spherical_harmonics_impl=impl, **kw)
    z = torch.zeros((1,) + grid.modal_shape, device=gpu_device)
    return sh._winds_handle(grid, z, z, grid.modal_shape)

  first = handle()
  assert handle() is first and handle(radius=2.0) is not first


# 12 and 200 fields: 4 and 8 a thread
@pytest.mark.parametrize('fields', [12, 200])
def test_modal_winds_are_rounded_once(gpu_device, fields):
  """FP32 fields: each result is the FP64 one rounded, whose error the polar winds
  amplify no further."""
  grid = sh.Grid.T85()
  gen = torch.Generator(device=gpu_device).manual_seed(3)
  mask = torch.as_tensor(grid.mask, device=gpu_device)
  a, b = (torch.randn((fields,) + grid.modal_shape, generator=gen, device=gpu_device) * mask
          for _ in range(2))
  handle = sh._winds_handle(grid, a, b, grid.modal_shape)
  a64, b64 = a.double(), b.double()
  exact = {0: sh.get_cos_lat_vector(a64, b64, grid),
           2: (grid.curl_cos_lat((a64, b64)), grid.div_cos_lat((a64, b64)))}
  for mode, refs in exact.items():
    got = sh._Winds.apply(a, b, handle, mode, True).double()
    for x, ref in zip((got[:fields], got[fields:]), refs):
      err = torch.where(mask, x - ref, 0.0).abs()  # below the triangle: not all written
      # half an ulp, and the FP64 terms' own rounding
      assert (err <= 2.0 ** -24 * ref.abs() + 1e-14 * ref.abs().max()).all(), mode
