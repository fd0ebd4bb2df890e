"""fem_grad_samples (the states the law check looks at) against torch's own
selection from all gradients: meshes of less than 48 points, of one list of 1024,
just past it, and of several; with NaN and infinite gradients; HEX27."""
import numpy as np
import pytest
import torch

from jax_fem_amd import materials
from jax_fem_amd._lib import check, ptr, stream_ptr
from jax_fem_amd.generate_mesh import Mesh, box_mesh, box_mesh_hex27
from jax_fem_amd.problem import Problem

pytestmark = pytest.mark.gpu


class _Law(Problem):
    def get_tensor_map(self):
        return materials.LinearElastic(E=1., nu=0.3) if self.vec[0] == 3 else materials.Poisson(k=1.)


@pytest.mark.parametrize('vec', [1, 3])
@pytest.mark.parametrize('second,n,bad', [(False, (1, 1, 1), 0), (False, (128, 1, 1), 0), (False, (43, 3, 1), 0),
                                          (False, (20, 21, 22), 0), (False, (20, 21, 22), 5), (True, (4, 3, 3), 0)])
def test_largest_gradients_and_spread_points(gpu, vec, second, n, bad):
    m = (box_mesh_hex27 if second else box_mesh)(*n, 1., 1., 1.)
    kw = dict(ele_type='HEX27', quadrature_order=4) if second else {}
    p = _Law(Mesh(m.points, m.cells_dict['hexahedron27' if second else 'hexahedron']), vec=vec, dim=3, **kw)
    dev = p.device()
    dm = dev.dm
    u = torch.randn(dev.n, dtype=torch.float64, device='cuda', generator=torch.Generator(device='cuda').manual_seed(2))
    if bad:
        u[7 * vec], u[100 * vec] = float('nan'), float('inf')
    G = dev.quad_grad(u)
    N = G.shape[0]
    k = min(N, 48)
    idx = torch.empty(2 * k, dtype=torch.int64, device='cuda')
    got = torch.empty((2 * k, vec, 3), dtype=torch.float64, device='cuda')
    ws = torch.empty(int(dev.L.fem_grad_samples_ws_bytes(dm.ref)), dtype=torch.uint8, device='cuda')
    check(dev.L.fem_grad_samples(dm.ref, ptr(u), k, k, ptr(idx), ptr(got), ptr(ws), stream_ptr()), 'fem_grad_samples')
    assert torch.equal(got.nan_to_num(), G[idx].nan_to_num())         # the same kernel arithmetic: bit for bit
    mag = G.reshape(N, -1).abs().amax(1)
    mag = torch.where(torch.isfinite(G.reshape(N, -1)).all(1), mag, torch.full_like(mag, -1.))
    assert len(torch.unique(idx[:k])) == k
    assert torch.equal(mag[idx[:k]], torch.topk(mag, k).values)
    want = np.linspace(0, N - 1, k)
    assert np.abs(idx[k:].cpu().numpy() - want).max() <= 1
