"""fem_grad_samples of a field at rest: all keys are exactly equal, so every selection, the
merging pass's among them, goes through all bytes and falls to the positions."""
import numpy as np
import pytest
import torch

from jax_fem_amd import materials
from jax_fem_amd._lib import check, ptr, stream_ptr
from jax_fem_amd.generate_mesh import Mesh, box_mesh
from jax_fem_amd.problem import Problem

pytestmark = pytest.mark.gpu


class _Law(Problem):
    def get_tensor_map(self):
        return materials.LinearElastic(E=1., nu=0.3)


@pytest.mark.parametrize('n', [(3, 2, 1), (40, 40, 31), (64, 64, 64)])   # one list, and merges of 8192 keys
def test_equal_keys(gpu, n):
    m = box_mesh(*n, 1., 1., 1.)
    dev = _Law(Mesh(m.points, m.cells_dict['hexahedron']), vec=3, dim=3).device()
    N = 8 * n[0] * n[1] * n[2]
    k = min(N, 48)
    u = torch.zeros(dev.n, dtype=torch.float64, device='cuda')
    idx = torch.full((2 * k,), -1, dtype=torch.int64, device='cuda')
    got = torch.full((2 * k, 9), 7., dtype=torch.float64, device='cuda')
    ws = torch.empty(int(dev.L.fem_grad_samples_ws_bytes(dev.dm.ref)), dtype=torch.uint8, device='cuda')
    check(dev.L.fem_grad_samples(dev.dm.ref, ptr(u), k, k, ptr(idx), ptr(got), ptr(ws), stream_ptr()), 'fem_grad_samples')
    i = idx.cpu().numpy()
    assert i.min() >= 0 and i.max() < N and len(np.unique(i[:k])) == k
    assert np.abs(i[k:] - np.linspace(0, N - 1, k)).max() <= 1
    assert float(got.abs().max()) == 0.
