"""fem_grad_samples where its lists take a merging pass of their own, with fewer points a
cell than a round of 256 takes, and with gradients that are all equal (the selection
then goes through every byte of the key and falls to the positions): against torch's
selection from all gradients, bit for bit (one arithmetic, no sums between points)."""
import pytest
import torch

from jax_fem_amd import materials
from jax_fem_amd._lib import check, ptr, stream_ptr
from jax_fem_amd.generate_mesh import Mesh, box_mesh, box_mesh_hex27
from jax_fem_amd.problem import Problem

pytestmark = pytest.mark.gpu


class _Law(Problem):
    def get_tensor_map(self):
        return materials.LinearElastic(E=1., nu=0.3)


@pytest.mark.parametrize('second,n,order,kind', [(False, (40, 40, 31), None, 'random'), (False, (64, 64, 64), None, 'random'),
                                                 (False, (31, 5, 3), 1, 'random'), (False, (9, 8, 7), 6, 'random'),
                                                 (True, (5, 5, 5), 2, 'random'), (False, (40, 40, 31), None, 'equal'),
                                                 (False, (5, 4, 3), None, 'zero')])
def test_selection(gpu, second, n, order, kind):
    m = (box_mesh_hex27 if second else box_mesh)(*n, 1., 1., 1.)
    kw = dict(quadrature_order=order) if order else {}
    p = _Law(Mesh(m.points, m.cells_dict['hexahedron27' if second else 'hexahedron']), vec=3, dim=3,
             ele_type='HEX27' if second else 'HEX8', **kw)
    dev = p.device()
    dm = dev.dm
    u = torch.randn(dev.n, dtype=torch.float64, device='cuda', generator=torch.Generator(device='cuda').manual_seed(2))
    if kind != 'random':
        u = torch.zeros_like(u) if kind == 'zero' else torch.ones_like(u)
    G = dev.quad_grad(u).reshape(-1, 9)
    if kind == 'equal':
        G = G * 0.
    N = G.shape[0]
    k = min(N, 48)
    idx = torch.full((2 * k,), -1, dtype=torch.int64, device='cuda')
    got = torch.empty((2 * k, 9), dtype=torch.float64, device='cuda')
    ws = torch.empty(int(dev.L.fem_grad_samples_ws_bytes(dm.ref)), dtype=torch.uint8, device='cuda')
    check(dev.L.fem_grad_samples(dm.ref, ptr(u), k, k, ptr(idx), ptr(got), ptr(ws), stream_ptr()), 'fem_grad_samples')
    assert int(idx.min()) >= 0 and int(idx.max()) < N and len(torch.unique(idx[:k])) == k
    if kind == 'random':
        assert torch.equal(got, G[idx])
        mag = G.abs().amax(1)
        assert torch.equal(mag[idx[:k]], torch.topk(mag, k).values)
    else:
        assert float(got.abs().max()) < 1e-12
