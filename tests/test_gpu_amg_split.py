"""AMG-CG whose level 0 reads the matrix (the plastic law at rest: no matrix-free products) at the
splits of its products: FP64 blocks and HEX27 rows (eight waves a slice), FP32 and FP16 blocks of
HEX8 (three and four), scalar rows of both; one slice, a last slice of one row, several slices.

The solve's own criterion bounds the result: the true residual with the assembled matrix is the
recursion's to about 1e-16 of |A| |x|, 1 % of rtol |b| at most."""
import pytest
import torch

from jax_fem_amd import _lib, materials
from jax_fem_amd.generate_mesh import Mesh, box_mesh, box_mesh_hex27
from jax_fem_amd.problem import Problem
from jax_fem_amd.solver import get_A, linear_config
from problems import isclose

pytestmark = pytest.mark.gpu


class _Heat(Problem):
    def get_tensor_map(self):
        return materials.Poisson(k=1.)


class _Plastic(Problem):
    def get_tensor_map(self):
        return materials.J2Plastic(E=1., nu=0.3, sig0=1e3)


@pytest.mark.parametrize('options', [dict(precision='fp64'), dict(precision='mixed'),
                                     dict(precision='mixed', level0='fp16'), dict(precision='mixed', outer='fp32')],
                         ids=['fp64', 'mixed', 'fp16', 'outer32'])
@pytest.mark.parametrize('ele,vec,n', [('HEX8', 3, (4, 4, 12)), ('HEX8', 3, (12, 12, 13)), ('HEX8', 1, (20, 20, 20)),
                                       ('HEX27', 3, (2, 2, 6)), ('HEX27', 3, (5, 6, 6)), ('HEX27', 1, (9, 9, 9))])
def test_every_split_solves_the_system(gpu, ele, vec, n, options):
    clamp = [[lambda x: isclose(x[0], 0.)] * vec, list(range(vec)), [lambda x: 0.] * vec]
    m = (box_mesh if ele == 'HEX8' else box_mesh_hex27)(*n, 1., 1., 1.)
    mesh = Mesh(m.points, m.cells_dict['hexahedron' if ele == 'HEX8' else 'hexahedron27'])
    p = (_Heat if vec == 1 else _Plastic)(mesh, vec=vec, dim=3, ele_type=ele, dirichlet_bc_info=clamp,
                                          **({} if ele == 'HEX8' else dict(quadrature_order=4)))
    if vec == 3:
        shape = (p.num_cells, p.fes[0].num_quads, 3, 3)
        p.internal_vars = [torch.zeros(shape, dtype=torch.float64, device='cuda') for _ in range(2)]
    dev = p.device()
    dev.prepare()
    b = torch.randn(dev.n, dtype=torch.float64, device='cuda',
                    generator=torch.Generator(device='cuda').manual_seed(4))
    b[dev.bc_dofs_long] = 0.
    cfg = linear_config({'amgx_solver': dict(tol=1e-8, atol=0., **options)})
    u = torch.zeros_like(b)
    dev.tangent(u, cfg['precision_code'])
    x, info = dev.solve(u, b, torch.zeros_like(b), cfg)
    assert info.status == _lib.FEM_OK and info.res_norm <= 1e-8 * info.b_norm
    assert torch.linalg.norm(b - get_A(p).spmv(x)) <= 1.01e-8 * torch.linalg.norm(b)
    assert torch.equal(x, dev.solve(u, b, torch.zeros_like(b), cfg)[0])
