"""Jacobi-PCG products of block rows and of long rows where the launch changes: FP32 blocks at 512
slices (eight and four waves), FP64 blocks beyond 768 (eight), HEX27 rows of either width (eight
waves, also where the direction has a kernel of its own), and sizes either side of the largest
matrices whose product forms the direction.

The plastic law at rest (the elastic tangent, but no matrix-free products).  The solve's own
criterion bounds each result: the true residual, formed with the assembled matrix, is the
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


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('ele,vec,n', [
    ('HEX8', 3, (31, 31, 31)), ('HEX8', 3, (31, 31, 32)),    # 512 and 528 slices
    ('HEX8', 3, (36, 36, 35)), ('HEX8', 3, (36, 36, 36)),    # 770 and 792
    ('HEX8', 3, (45, 45, 45)),                               # FP32 past 100 MB
    ('HEX27', 1, (20, 20, 20)), ('HEX27', 3, (9, 10, 11)),
    ('HEX27', 1, (23, 23, 23)),                              # FP64 past 45 MB
    ('HEX27', 3, (20, 20, 21))])                             # past 240 MB (FP64), of FP32 below 180
def test_products_of_every_form_solve_the_system(gpu, ele, vec, n, precision):
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
    its = {}
    for check_every in (16, 1):
        cfg = linear_config({'jax_solver': dict(precision=precision, tol=1e-8, atol=0., check_every=check_every)})
        u = torch.zeros_like(b)
        dev.tangent(u, cfg['precision_code'])
        x, info = dev.solve(u, b, torch.zeros_like(b), cfg)
        assert info.status == _lib.FEM_OK and info.res_norm <= 1e-8 * info.b_norm
        its[check_every] = info.iterations
        if precision == 'fp64':
            assert torch.linalg.norm(b - get_A(p).spmv(x)) <= 1.01e-8 * torch.linalg.norm(b)
        again = dev.solve(u, b, torch.zeros_like(b), cfg)[0]
        assert torch.equal(x, again)
    if precision == 'fp64':
        assert abs(its[16] - its[1]) <= 2 + 0.03 * its[16], its
