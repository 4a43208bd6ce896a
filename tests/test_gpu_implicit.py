"""Implicit solve and terms with one and with two 16-column tiles a wave."""
import pytest
import torch

from dinosaur_amd import workloads

pytestmark = pytest.mark.gpu


# T21 has 62 tiles a member: 264 members stay below the 8 blocks per CU of a 256-CU
# card up to which a wave takes one tile, 265 are above (two tiles, the last block
# with an odd rest); T42 (234 tiles, the last with 12 columns) likewise at 70 and 71.
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('name,K,members', [('T21', 3, 264), ('T21', 3, 265), ('T42', 5, 70),
                                            ('T42', 5, 71)])
@pytest.mark.parametrize('fn', ['solve', 'terms', 'solve_adjoint', 'terms_adjoint',
                                'terms_adjoint_accumulate'])
def test_members_of_a_batch_equal_members_alone(fn, name, K, members, dtype, gpu_device):
  eq, _, coords, _ = workloads.build_primitive(name, K, moist=False, members=1, dtype=dtype,
                                               device=gpu_device)
  gen = torch.Generator(device=gpu_device).manual_seed(K + members)
  mask = torch.as_tensor(coords.horizontal.mask, device=gpu_device)

  def fields():
    return [torch.randn(members, k, *coords.horizontal.modal_shape, device=gpu_device, dtype=dtype,
                        generator=gen) * mask for k in (K, K, 1)]

  x, batch = fields(), fields()
  alone = [t.clone() for t in batch]
  call = lambda n, src, dst: eq._implicit.apply_into('dino_implicit_' + fn, 0.02, n, *src, *dst)
  call(members, x, batch)
  for e in range(members):
    call(1, [t[e] for t in x], [t[e] for t in alone])
  for a, b in zip(batch, alone):
    assert torch.equal(a, b)  # the same operations in the same order
