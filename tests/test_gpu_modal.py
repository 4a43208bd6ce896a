"""Modal kernels of one explicit evaluation with one, two and four levels a thread."""
import ctypes

import pytest
import torch

from dinosaur_amd import _lib, primitive_equations as pe, spherical_harmonic as sh

pytestmark = pytest.mark.gpu


# T21 has 989 entries a level and T85 14877: 24 members of T21 L11 are on the one-level
# side of 2^18 entries, 25 on the two-level side (an odd rest of 11), 173 members of T85
# L13 on the two-level side of 2^25 and 174 on the four-level side (a rest of one).
# Every member equals the member alone, a thread a level: the sums are the same.
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
# Without tracers the epilogue and the prep's adjoint change at 2^20 (FP32) and 2^22 (FP64):
# 5 and 6, 21 and 22 members of T85 L13.
@pytest.mark.parametrize('name,K,members,check,tracers', [
    ('T21', 11, 24, range(24), 1), ('T21', 11, 25, range(25), 1),
    ('T85', 13, 173, (0, 100, 172), 1), ('T85', 13, 174, (0, 100, 173), 1),
    ('T85', 13, 5, (0, 4), 0), ('T85', 13, 6, (0, 5), 0), ('T85', 13, 21, (0, 20), 0),
    ('T85', 13, 22, (0, 21), 0)])
@pytest.mark.parametrize('fn', ['prep', 'prep_adjoint', 'epilogue', 'epilogue_adjoint'])
def test_members_of_a_batch_equal_members_alone(fn, name, K, members, check, tracers, dtype,
                                                gpu_device):
  grid = getattr(sh.Grid, name)()
  R, L = grid.modal_shape
  h = pe.modal_handle(grid, K, tracers, tracers - 1, 9.8, gpu_device)
  levels = {'state': [K, K, K, 1, K], 'prep': [K] * 6 + [1, 1, 1, K, K],
            'epilogue': [K] * 6 + [1] + [K] * 5}
  if not tracers:
    levels = {'state': [K, K, K, 1], 'prep': [K] * 5 + [1, 1], 'epilogue': [K] * 6 + [1]}
  groups = ('state', 'prep', 'epilogue')
  src, dst = {'prep': (0, 1), 'prep_adjoint': (1, 0), 'epilogue': (2, 0),
              'epilogue_adjoint': (0, 2)}[fn]
  for which in (src, dst):
    assert _lib.lib().dino_modal_fields(h.handle, members, which) == members * sum(
        levels[groups[which]])
  gen = torch.Generator(device=gpu_device).manual_seed(K)

  def call(n, x):
    out = torch.zeros(n * sum(levels[groups[dst]]), R, L, device=gpu_device, dtype=dtype)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    code = _lib.DINO_F64 if dtype == torch.float64 else _lib.DINO_F32
    _lib.check(getattr(_lib.lib(), 'dino_modal_' + fn)(h.handle, ptr(x), None, ptr(out), n, code,
                                                       stream), fn)
    return out

  def member(x, which, e):
    parts, o = [], 0
    for lev in levels[groups[which]]:
      parts.append(x[o + e * lev:o + (e + 1) * lev])
      o += members * lev
    return torch.cat(parts)

  x = torch.randn(members * sum(levels[groups[src]]), R, L, device=gpu_device, dtype=dtype,
                  generator=gen)
  batch = call(members, x)
  for e in check:
    assert torch.equal(member(batch, dst, e), call(1, member(x, src, e)))
