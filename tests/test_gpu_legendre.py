"""Legendre kernels at every latitude count where their tiles change: node
tiles and blocks of 16 / 128 nodes, the 4- and 8-wave forms, the two-wave
strips above 128 northern nodes, the tiled kernels above 512; batches around
the 16-, 64- and 128-row groups; odd latitude counts (the equator counts
once) and buffers off 16-byte alignment; against the plan's own table in FP64.

Tolerance: sums of n products of rounded operands, 4 u sqrt(n) normwise, with
u = 2^-24 (FP32), 2^-53 (FP64); split BF16 keeps 16 bits of each operand and
drops the product of the low parts, 4 * 2^-16.
"""
import ctypes

import numpy as np
import pytest
import torch

from dinosaur_amd import _lib
from dinosaur_amd import spherical_harmonic as sh

pytestmark = pytest.mark.gpu

NODES = [1, 5, 16, 17, 32, 33, 48, 64, 65, 80, 90, 96, 97, 128, 129, 144, 160, 192, 193, 256, 257,
         272, 320, 321, 400, 512, 513]


def _reference(plan, forward, x):
  """FP64 sums with the plan's folded table; x (B, R, J) or (B, R, L)."""
  M, L, J = plan.M, plan.L, plan.J
  jh = (J + 1) // 2
  table, pos = plan.folded_table(), 0
  out = np.zeros((x.shape[0], plan.R, L if forward else J))
  for m in range(M):
    rows = table[pos:pos + (L - m) * jh].reshape(L - m, jh)
    pos += (L - m) * jh
    sign = np.where(np.arange(L - m) % 2 == 0, 1.0, -1.0)[:, None]
    p = np.zeros((L - m, J))
    p[:, :jh] = (rows * sign)[:, ::-1]
    p[:, J - jh:] = rows
    for r in ([0] if m == 0 else [2 * m - 1, 2 * m]):
      if forward:
        out[:, r, m:] = x[:, r] @ p.T
      else:
        out[:, r] = x[:, r, m:] @ p
  return out


@pytest.mark.parametrize('odd', [0, 1])
@pytest.mark.parametrize('nodes', NODES)
def test_legendre_matches_table(gpu_device, nodes, odd):
  J = 2 * nodes - odd
  lib = _lib.lib()
  p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
  stream = ctypes.c_void_p(torch.cuda.current_stream(gpu_device).cuda_stream)
  rng = np.random.default_rng(J)
  # 75 degrees: three 32-degree tiles with zeros below the first
  M, L = 21, 75
  plan = sh.get_plan(M, L, 2 * M, J, 'gauss', gpu_device)
  cases = [(_lib.DINO_F32, _lib.PREC_NATIVE, 4 * 2.0 ** -24 * max(L, nodes) ** 0.5),
           (_lib.DINO_F32, _lib.PREC_BF16X3, 4 * 2.0 ** -16),
           (_lib.DINO_F64, _lib.PREC_NATIVE, 4 * 2.0 ** -53 * max(L, nodes) ** 0.5)]
  for B, skew, sched in ((3, 0, 0), (8, 1, 0), (37, 0, _lib.SCHED_MPAIRED), (66, 0, 0)):
    print('[test] legendre', J, B, skew, flush=True)
    f = rng.standard_normal((B, plan.R, J))
    x = rng.standard_normal((B, plan.R, L))
    for stage in (_lib.STAGE_LEGENDRE_INVERSE, _lib.STAGE_LEGENDRE_FORWARD):
      plan.set_schedule(stage, sched)
    for code, prec, tol in cases:
      dtype = torch.float32 if code == _lib.DINO_F32 else torch.float64

      def skewed(a):
        buf = torch.full((a.size + skew + 8,), 7.0, dtype=dtype, device=gpu_device)
        view = buf[skew:skew + a.size].view(a.shape)
        view.copy_(torch.as_tensor(a, device=gpu_device))
        return buf, view

      for forward in (True, False):
        src, dst = (f, x) if forward else (x, f)
        _, xin = skewed(src)
        buf, out = skewed(np.zeros_like(dst))
        fn = lib.dino_legendre_forward if forward else lib.dino_legendre_inverse
        _lib.check(fn(plan.handle, p(xin), p(out), B, code, prec, stream))
        ref = _reference(plan, forward, xin.double().cpu().numpy())
        got = out.double().cpu().numpy()
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err <= tol, (forward, code, prec, B, skew, err)
        assert (buf[:skew] == 7.0).all() and (buf[skew + dst.size:] == 7.0).all()
        if forward:  # written only from the first tile's degrees on, the triangle whole
          buf, out = skewed(np.full_like(dst, 3.0))
          _lib.check(fn(plan.handle, p(xin), p(out), B, code, prec | _lib.SHT_TRIANGLE_ONLY,
                        stream))
          tri = np.arange(L) >= (np.arange(plan.R)[:, None] + 1) // 2
          got = out.double().cpu().numpy() * tri
          assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), (code, prec, B, skew)
          assert (buf[:skew] == 7.0).all() and (buf[skew + dst.size:] == 7.0).all()
  for stage in (_lib.STAGE_LEGENDRE_INVERSE, _lib.STAGE_LEGENDRE_FORWARD):
    plan.set_schedule(stage, 0)


# Northern nodes of each forward kernel: row-resident, split, tiled; FP64 on the
# matrix cores (4, 8, 16 node groups) and in FMA tiles (257 up).
@pytest.mark.parametrize('nodes', [16, 65, 129, 256, 257, 513])
@pytest.mark.parametrize('code,prec', [(_lib.DINO_F32, _lib.PREC_NATIVE),
                                       (_lib.DINO_F32, _lib.PREC_BF16X3),
                                       (_lib.DINO_F64, _lib.PREC_NATIVE)])
def test_triangle_only_rows_are_whole_from_their_first_tile(gpu_device, nodes, code, prec):
  M, L, J = 40, 75, 2 * nodes
  print('[test] triangle only', nodes, code, prec, flush=True)
  plan = sh.get_plan(M, L, 2 * M, J, 'gauss', gpu_device)
  dtype = torch.float32 if code == _lib.DINO_F32 else torch.float64
  lib, p = _lib.lib(), lambda t: ctypes.c_void_p(t.data_ptr())
  stream = ctypes.c_void_p(torch.cuda.current_stream(gpu_device).cuda_stream)
  m = (torch.arange(plan.R, device=gpu_device)[:, None] + 1) // 2
  start = (L - 32 * ((L - m + 31) // 32)).clamp(min=0)
  l = torch.arange(L, device=gpu_device)
  for B in (1, 40):
    x = torch.randn((B, plan.R, J), dtype=dtype, device=gpu_device)
    whole, part = (torch.full((B, plan.R, L), float('nan'), dtype=dtype, device=gpu_device)
                   for _ in range(2))
    for out, flag in ((whole, 0), (part, _lib.SHT_TRIANGLE_ONLY)):
      _lib.check(lib.dino_legendre_forward(plan.handle, p(x), p(out), B, code, prec | flag,
                                           stream))
    assert (whole[:, l < m] == 0).all()
    assert part[:, l >= start].equal(whole[:, l >= start])
