"""Mixed-precision Jacobi-PCG of block rows and long rows, at the sizes where the launch changes,
against the assembled FP64 matrix: the true residual, which the solver forms without it, is that
of the matrix to about 1e-16 of |A| |x|, 1 % of rtol |b| at most."""
import pytest
import torch

from jax_fem_amd import _lib, materials
from jax_fem_amd.generate_mesh import Mesh, box_mesh, box_mesh_hex27
from jax_fem_amd.problem import Problem
from jax_fem_amd.solver import linear_config
from problems import isclose

pytestmark = pytest.mark.gpu


class _Heat(Problem):
    def get_tensor_map(self):
        return materials.Poisson(k=1.)


class _Plastic(Problem):
    def get_tensor_map(self):
        return materials.J2Plastic(E=1., nu=0.3, sig0=1e3)


@pytest.mark.parametrize('check_every', [16, 1])
@pytest.mark.parametrize('ele,vec,n', [('HEX8', 3, (12, 12, 13)), ('HEX8', 3, (31, 31, 31)), ('HEX8', 3, (31, 31, 32)),
                                       ('HEX8', 3, (45, 45, 45)), ('HEX8', 1, (10, 10, 10)), ('HEX27', 1, (12, 12, 12)),
                                       ('HEX27', 3, (9, 10, 11))])
def test_true_residual(gpu, ele, vec, n, check_every):
    m = (box_mesh if ele == 'HEX8' else box_mesh_hex27)(*n, 1., 1., 1.)
    mesh = Mesh(m.points, m.cells_dict['hexahedron' if ele == 'HEX8' else 'hexahedron27'])
    clamp = [[lambda x: isclose(x[0], 0.)] * vec, list(range(vec)), [lambda x: 0.] * vec]
    p = (_Heat if vec == 1 else _Plastic)(mesh, vec=vec, dim=3, ele_type=ele, dirichlet_bc_info=clamp,
                                          **({} if ele == 'HEX8' else dict(quadrature_order=4)))
    if vec == 3:
        shape = (p.num_cells, p.fes[0].num_quads, 3, 3)
        p.internal_vars = [torch.zeros(shape, dtype=torch.float64, device='cuda') for _ in range(2)]
    dev = p.device()
    dev.prepare()
    b = torch.randn(dev.n, dtype=torch.float64, device='cuda', generator=torch.Generator(device='cuda').manual_seed(4))
    b[dev.bc_dofs_long] = 0.
    u = torch.zeros_like(b)
    cfg = linear_config({'jax_solver': dict(precision='mixed', tol=1e-8, atol=0., check_every=check_every)})
    dev.tangent(u, cfg['precision_code'])
    x, info = dev.solve(u, b, torch.zeros_like(b), cfg)
    assert info.status == _lib.FEM_OK and info.res_norm <= 1e-8 * info.b_norm
    dev.tangent(u, _lib.FEM_F64)
    assert torch.linalg.norm(b - dev.spmv(x)) <= 1.01e-8 * torch.linalg.norm(b)
