"""Forward Legendre sums of a field dominated by its mean: the coefficients of every
other degree are what is left of sums that cancel, so an order of summation whose
partial sums stay large shows there and not in a norm of the whole result."""
import ctypes

import numpy as np
import pytest
import torch

from dinosaur_amd import _lib, spherical_harmonic as sh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('J', [320, 384, 512, 640, 800, 1000])
@pytest.mark.parametrize('B', [3, 40])
def test_partial_sums_stay_small(gpu_device, J, B):
  M, L = 3, J // 2
  plan = sh.get_plan(M, L, 8, J, 'gauss', gpu_device)
  jh = J // 2
  rows = plan.folded_table()[:L * jh].reshape(L, jh)  # m = 0, equator to pole
  rng = np.random.default_rng(J)
  scale = rng.uniform(0.5, 2.0, B)
  half = (np.polynomial.legendre.leggauss(J)[1][jh:] * rows[0])[None] * scale[:, None]
  x = np.zeros((B, plan.R, J), np.float32)
  x[:, 0] = np.concatenate([half[:, ::-1], half], axis=1)
  xin = torch.as_tensor(x, device=gpu_device)
  out = torch.zeros(B, plan.R, L, device=gpu_device)
  ptr = lambda t: ctypes.c_void_p(t.data_ptr())
  stream = ctypes.c_void_p(torch.cuda.current_stream(gpu_device).cuda_stream)
  _lib.check(_lib.lib().dino_legendre_forward(plan.handle, ptr(xin), ptr(out), B, _lib.DINO_F32,
                                              _lib.PREC_NATIVE, stream), 'forward')
  # even degrees; terms as the kernel forms them (folded rows and table in FP32)
  folded = (x[:, 0, jh:] + x[:, 0, jh - 1::-1]).astype(np.float64)
  terms = folded[:, None] * rows[0::2].astype(np.float32).astype(np.float64)
  err2 = (out[:, 0, 0::2].double().cpu().numpy() - terms.sum(-1)) ** 2
  # Partial sums over neighbouring nodes fall as 1 / l, and the roundings with them:
  # about half an octave further up (0.3 to 0.6 in a simulation of one chain and of
  # two halves).  Groups of 16 nodes taken in turn by two chains are a square wave
  # of 32 nodes, whose partial sums peak at its alias l = J / 16 (1.6 to 3.7).
  band = lambda c: err2[:, int(0.75 * c) // 2:int(1.3 * c) // 2 + 1].mean() ** 0.5  # noqa: E731
  ratio = band(J / 16) / band(J / 32)
  print('J', J, 'B', B, 'ratio', ratio, flush=True)
  assert ratio < 1
