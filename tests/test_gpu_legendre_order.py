"""Row-resident Legendre kernels with several row blocks: the XCD launch order, the
96-row blocks of large tables, and both m orders, against pieces of one row block."""
import ctypes

import pytest
import torch

from dinosaur_amd import _lib, spherical_harmonic as sh

pytestmark = pytest.mark.gpu


# 8 XCDs take m in turn: M = 107 and 341 leave a rest, 256 none.  Inverse, FP32: 448 and
# 449 fields (14 and 15 row blocks) lie on both sides of its line; the table of 341 x
# 342 x 256 values exceeds 32 MB, so 33 to 48 fields take 96 rows a block.
@pytest.mark.parametrize('prec', [_lib.PREC_NATIVE, _lib.PREC_BF16X3])
@pytest.mark.parametrize('sched', [0, _lib.SCHED_MPAIRED])
@pytest.mark.parametrize('M,L,I,J,batches', [
    (107, 108, 320, 160, (33, 448, 449)), (256, 257, 512, 256, (40, 100)),
    (341, 342, 1024, 512, (32, 33, 48, 49, 100))])
def test_batch_equals_its_pieces(gpu_device, M, L, I, J, batches, sched, prec):
  plan = sh.get_plan(M, L, I, J, 'gauss', gpu_device)
  lib = _lib.lib()
  stream = ctypes.c_void_p(torch.cuda.current_stream(gpu_device).cuda_stream)
  gen = torch.Generator(device=gpu_device).manual_seed(M)
  for forward in (True, False):
    fn = lib.dino_legendre_forward if forward else lib.dino_legendre_inverse
    stage = _lib.STAGE_LEGENDRE_FORWARD if forward else _lib.STAGE_LEGENDRE_INVERSE
    cols = (J, L) if forward else (L, J)

    def call(x):
      out = torch.full((x.shape[0], plan.R, cols[1]), 7.0, device=gpu_device)
      _lib.check(fn(plan.handle, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(out.data_ptr()),
                    x.shape[0], _lib.DINO_F32, prec, stream), 'legendre')
      return out

    for B in batches:
      x = torch.randn(B, plan.R, cols[0], device=gpu_device, generator=gen)
      plan.set_schedule(stage, sched)
      try:
        whole = call(x)
      finally:
        plan.set_schedule(stage, 0)
      pieces = torch.cat([call(part) for part in x.split(16)])
      # a row's sums run in the same order whichever block holds it
      assert torch.equal(whole, pieces), (forward, B)


# FP64: T85-sized with 32- and 64-node blocks (forward: split over the degree tiles, and
# several tiles a block), 128 nodes on both sides of the FMA tiles' line (512 row blocks:
# 64 fields), 160 nodes likewise (8 and 32 fields), 24 nodes, and 257 nodes (FMA forward).
@pytest.mark.parametrize('M,L,I,J,batches', [
    (32, 33, 96, 48, (40, 700)), (86, 87, 256, 128, (100, 400)), (256, 257, 512, 256, (40, 100)),
    (214, 215, 640, 320, (8, 32, 40)), (60, 75, 180, 513, (9, 80))])
def test_fp64_batch_equals_its_pieces(gpu_device, M, L, I, J, batches):
  plan = sh.get_plan(M, L, I, J, 'gauss', gpu_device)
  lib = _lib.lib()
  stream = ctypes.c_void_p(torch.cuda.current_stream(gpu_device).cuda_stream)
  gen = torch.Generator(device=gpu_device).manual_seed(M)
  table, jh = torch.as_tensor(plan.folded_table(), device=gpu_device), (J + 1) // 2
  for forward in (True, False):
    fn = lib.dino_legendre_forward if forward else lib.dino_legendre_inverse
    cols = (J, L) if forward else (L, J)

    def call(x):
      out = torch.full((x.shape[0], plan.R, cols[1]), 7.0, device=gpu_device, dtype=x.dtype)
      _lib.check(fn(plan.handle, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(out.data_ptr()),
                    x.shape[0], _lib.DINO_F64, _lib.PREC_NATIVE, stream), 'legendre')
      return out

    for B in batches:
      print('[test] fp64 legendre order', M, J, B, forward, flush=True)
      x = torch.randn(B, plan.R, cols[0], device=gpu_device, generator=gen, dtype=torch.float64)
      whole = call(x)
      # whichever kernel a batch takes adds in the same order
      assert torch.equal(whole, torch.cat([call(part) for part in x.split(5)])), (forward, B)
      # rows of some m against the plan's table: sums of n products, 4 u sqrt(n)
      for m in (0, 1, M // 2, M - 1):
        pos = sum((L - k) * jh for k in range(m))
        p = table[pos:pos + (L - m) * jh].view(L - m, jh)
        sign = 1.0 - 2.0 * (torch.arange(L - m, device=gpu_device) % 2)[:, None]
        full = torch.zeros((L - m, J), device=gpu_device, dtype=torch.float64)
        full[:, :jh] = (p * sign).flip(1)
        full[:, J - jh:] = p
        r = 0 if m == 0 else 2 * m
        ref = x[:, r] @ full.T if forward else x[:, r, m:] @ full
        got = whole[:, r, m:] if forward else whole[:, r]
        assert (got - ref).norm() <= 4 * 2.0 ** -53 * max(L, J) ** 0.5 * ref.norm(), (forward, B, m)
