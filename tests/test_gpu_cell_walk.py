"""Element kernels whose workgroups walk the mesh: a mesh of more cells than the grid
takes in one trip, against itself with its cells in the opposite order (each cell's
result must not depend on the trip it is formed in; the sums inside a cell run in the
same order, so the results are equal bit for bit)."""
import pytest
import torch

from jax_fem_amd import _lib, materials as M
from jax_fem_amd._lib import check, ptr, stream_ptr
from jax_fem_amd.generate_mesh import Mesh, box_mesh, box_mesh_hex27
from jax_fem_amd.problem import Problem

pytestmark = pytest.mark.gpu


class _Law(Problem):
    def get_tensor_map(self):
        return M.SIMPElastic(E0=1., Emin=1e-3, nu=0.3, penal=3.)


@pytest.mark.parametrize('second,n,order', [(True, (12, 12, 13), 4), (False, (19, 19, 19), 4)])
def test_cells_in_either_order(gpu, second, n, order):
    m = (box_mesh_hex27 if second else box_mesh)(*n, 1., 1., 1.)
    cells = m.cells_dict['hexahedron27' if second else 'hexahedron']
    outs = []
    for flip in (False, True):
        p = _Law(Mesh(m.points, cells[::-1].copy() if flip else cells), vec=3, dim=3,
                 ele_type='HEX27' if second else 'HEX8', quadrature_order=order)
        gen = torch.Generator(device='cuda').manual_seed(4)
        rand = lambda *s: torch.rand(s, dtype=torch.float64, device='cuda', generator=gen)
        C, Q, N = p.num_cells, p.fes[0].num_quads, p.fes[0].num_nodes
        theta, mass = 0.3 + rand(C, Q), rand(C, Q, 3)
        u, lam = rand(p.fes[0].num_total_dofs), rand(p.fes[0].num_total_dofs)
        if flip:
            theta, mass = theta.flip(0).contiguous(), mass.flip(0).contiguous()
        p.internal_vars = [theta]
        dev = p.device()
        dev.prepare()
        dm, L, s = dev.dm, dev.L, stream_ptr()
        load, lq, g = torch.empty((C, N, 3), dtype=torch.float64, device='cuda'), torch.empty_like(mass), torch.empty_like(theta)
        check(L.fem_cell_load(dm.ref, ptr(mass), ptr(load), s), 'load')
        check(L.fem_cell_load_adjoint(dm.ref, ptr(lam), ptr(lq), s), 'load adjoint')
        check(L.fem_cell_adjoint(dm.ref, dev.mref, ptr(u), ptr(lam), ptr(g), s), 'adjoint')
        Ke = dev.cell_tangents(u, faces=False).reshape(C, -1)
        G = dev.quad_grad(u).reshape(C, -1)
        outs.append([t.flip(0) if flip else t for t in (load, lq, g, Ke, G)])
    for a, b in zip(*outs):
        assert float(a.abs().max()) > 0. and torch.equal(a, b)
