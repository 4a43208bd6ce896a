"""Longitude transform kernels at every kind of length: powers of two, lengths
with factors 2, 3, 5, 7 (mixed-radix FFT) and lengths with larger prime
factors, at latitude counts that leave partial tiles and unaligned rows,
against numpy's FP64 FFT.

Tolerance: an FFT or direct sum of I terms in a type of unit roundoff u is
within about u log2(I) (FFT) or u sqrt(I) (direct sum of random terms) of the
exact rows, normwise; 4 u sqrt(I) bounds both with room.
"""
import ctypes

import numpy as np
import pytest
import torch

from dinosaur_amd import _lib
from dinosaur_amd import spherical_harmonic as sh

pytestmark = pytest.mark.gpu

# (longitudes, wavenumbers, latitudes)
SHAPES = [
    (8, 3, 5), (12, 6, 4), (15, 8, 7), (48, 16, 24), (49, 25, 20), (70, 22, 33), (96, 32, 48),
    (105, 53, 52), (192, 96, 96), (243, 100, 31), (320, 107, 160), (360, 120, 180),
    (360, 180, 90), (375, 125, 36), (640, 214, 64), (1280, 640, 20), (1281, 600, 12),
    (2560, 1280, 9), (4096, 2048, 4), (64, 22, 32), (512, 256, 36), (1024, 341, 10),
    (2048, 1000, 6), (11, 6, 3), (67, 22, 34), (268, 89, 134), (341, 170, 171), (511, 170, 256),
    (127, 64, 64), (202, 101, 16), (583, 291, 40), (9, 1, 6),
    # the last smooth lengths of the matrix cores and the first of the mixed-radix FFT
    (60, 20, 30), (63, 32, 31), (70, 35, 9), (9, 5, 3), (45, 23, 23), (45, 1, 22),
]


def _rows(x, M):
  """Fourier rows (..., 2M-1, J) of nodal values (..., I, J), FP64."""
  spec = np.fft.rfft(x, axis=-2)[..., :M, :]
  out = np.zeros(x.shape[:-2] + (2 * M - 1, x.shape[-1]))
  out[..., 0, :] = spec[..., 0, :].real / np.sqrt(2 * np.pi)
  out[..., 1::2, :] = spec[..., 1:, :].real / np.sqrt(np.pi)
  out[..., 2::2, :] = -spec[..., 1:, :].imag / np.sqrt(np.pi)
  return out


def _nodal(g, I):
  """Values (..., I, J) of Fourier rows (..., 2M-1, J), FP64."""
  M = (g.shape[-2] + 1) // 2
  spec = np.zeros(g.shape[:-2] + (I // 2 + 1, g.shape[-1]), complex)
  spec[..., 0, :] = g[..., 0, :] / np.sqrt(2 * np.pi)
  spec[..., 1:M, :] = (g[..., 1::2, :] - 1j * g[..., 2::2, :]) / (2 * np.sqrt(np.pi))
  return np.fft.irfft(spec, n=I, axis=-2) * I


@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('shape', SHAPES)
def test_dft_matches_numpy(gpu_device, shape, dtype):
  I, M, J = shape
  print('[test] dft', shape, dtype, flush=True)
  lib = _lib.lib()
  plan = sh.get_plan(M, M + 1, I, J, 'gauss', gpu_device)
  code = _lib.DINO_F32 if dtype == torch.float32 else _lib.DINO_F64
  w = 2 * np.pi / I * plan.nodes()[1]
  rng = np.random.default_rng(I + J)
  tol = 4 * np.sqrt(I) * (2.0 ** -24 if dtype == torch.float32 else 2.0 ** -53)
  p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
  stream = ctypes.c_void_p(torch.cuda.current_stream(gpu_device).cuda_stream)
  # the second pass starts the buffers off 16-byte alignment
  if dtype == torch.float64 and I > 2730:  # beyond every FP64 kernel
    buf = torch.zeros((1, I, J), dtype=dtype, device=gpu_device)
    rc = lib.dino_dft_forward(plan.handle, p(buf), p(torch.zeros_like(buf)), 1, code, 0, stream)
    assert rc == _lib.DINO_EINVAL
    return
  for B, skew in ((3, 0), (2, 1)):
    x = torch.as_tensor(rng.standard_normal((B, I, J)), device=gpu_device).to(dtype)
    g = torch.as_tensor(rng.standard_normal((B, 2 * M - 1, J)), device=gpu_device).to(dtype)

    def skewed(t):
      buf = torch.empty(t.numel() + skew + 8, dtype=dtype, device=gpu_device).fill_(7.0)
      view = buf[skew:skew + t.numel()].view(t.shape)
      return buf, view

    for weighted in (0, 1):
      xin, out = skewed(x)[1], skewed(g)
      xin.copy_(x)
      _lib.check(lib.dino_dft_forward(plan.handle, p(xin), p(out[1]), B, code, weighted, stream))
      ref = _rows(x.double().cpu().numpy() * (w if weighted else 1.0), M)
      got = out[1].double().cpu().numpy()
      assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), ('forward', weighted, skew)
      assert (out[0][skew + g.numel():] == 7.0).all() and (out[0][:skew] == 7.0).all()
      gin, out = skewed(g)[1], skewed(x)
      gin.copy_(g)
      _lib.check(lib.dino_dft_inverse(plan.handle, p(gin), p(out[1]), B, code, weighted, stream))
      ref = _nodal(g.double().cpu().numpy(), I) * (w if weighted else 1.0)
      got = out[1].double().cpu().numpy()
      assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), ('inverse', weighted, skew)
      assert (out[0][skew + x.numel():] == 7.0).all() and (out[0][:skew] == 7.0).all()


# Kernels: per-tile FFT, persistent FFT (FP32), folded DFT, mixed-radix FFT, direct DFT;
# (9, 1, 6) the direct one of short lengths.
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('shape', [(64, 22, 32), (512, 170, 256), (128, 43, 64), (67, 22, 34),
                                   (320, 107, 160), (583, 291, 40), (9, 1, 6)])
def test_secant_weights(gpu_device, shape, dtype):
  """DINO_SHT_SEC_LAT: nodal values over cos(lat) after an inverse and before a forward
  transform, and in both adjoints: one rounding of the weight and one of the product
  more than the transform without it."""
  I, M, J = shape
  L = M + 1
  plan = sh.get_plan(M, L, I, J, 'gauss', gpu_device)
  print('[test] secant weights', shape, dtype, flush=True)
  sec = torch.as_tensor(1 / np.sqrt(1 - plan.nodes()[0] ** 2), device=gpu_device)
  tol = 8 * np.sqrt(max(I, J)) * (2.0 ** -24 if dtype == torch.float32 else 2.0 ** -53)
  gen = torch.Generator(device=gpu_device).manual_seed(I)
  x = torch.randn((5, I, J), generator=gen, device=gpu_device, dtype=torch.float64).to(dtype)
  m = torch.randn((5, 2 * M - 1, L), generator=gen, device=gpu_device,
                  dtype=torch.float64).to(dtype)
  m = m * (torch.arange(L, device=gpu_device) >= (torch.arange(2 * M - 1, device=gpu_device)[:, None]
                                                  + 1) // 2)
  scaled = lambda t: (t.double() * sec).to(dtype)  # noqa: E731
  call = lambda name, src, tail, flag: sh.sht_call(name, plan, src, tail, flag).double()  # noqa: E731
  for name, src, tail in (('dino_sht_inverse', m, (I, J)), ('dino_sht_forward_adjoint', m, (I, J)),
                          ('dino_sht_forward', x, (2 * M - 1, L)),
                          ('dino_sht_inverse_adjoint', x, (2 * M - 1, L))):
    got = call(name, src, tail, _lib.SHT_SEC_LAT)
    ref = call(name, src, tail, 0) * sec if src is m else call(name, scaled(src), tail, 0)
    assert (got - ref).norm() <= tol * ref.norm(), name
