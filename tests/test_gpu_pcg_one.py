"""Jacobi-PCG of small scalar systems in one workgroup (up to 22 slices, 1408 rows): at the
sizes where slices, the register-held part and the limit end, FP64 and mixed precision,
against the assembled matrix and a dense solve.

Tolerances: the solver's own criterion (true residual <= 1e-11 |b|), and against a dense
FP64 solve 1e-11 times the condition number (below 1e4 here), 1e-7."""
import numpy as np
import pytest
import torch

from jax_fem_amd import materials
from jax_fem_amd.generate_mesh import Mesh, box_mesh
from jax_fem_amd.problem import Problem
from jax_fem_amd.solver import solver
from problems import isclose

pytestmark = pytest.mark.gpu


class _Source(Problem):
    def get_tensor_map(self):
        return materials.Poisson(k=2.)

    def get_mass_map(self):
        return lambda u, x: torch.stack([-3. * x[0] + x[1] * x[2]])


def _mesh(kind):
    m = box_mesh(*kind, 1., 1., 1.)
    return Mesh(m.points, m.cells_dict['hexahedron'])


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('kind', [(1, 1, 1), (3, 3, 3), (4, 4, 3), (15, 15, 3), (16, 15, 3), (10, 10, 10), (15, 10, 7), (21, 15, 3), (21, 15, 4)])
def test_small_systems(gpu, kind, precision):
    p = _Source(_mesh(kind), vec=1, dim=3, dirichlet_bc_info=[[lambda x: isclose(x[0], 0.)], [0], [lambda x: 0.5]])
    opts = {'jax_solver': {'precision': precision, 'tol': 1e-11, 'atol': 0.}}
    u = solver(p, solver_options=opts)[0].reshape(-1)
    dev = p.device()
    st = p._solve_stats['linear'][0] if isinstance(p._solve_stats['linear'], list) else p._solve_stats['linear']
    dev.tangent(torch.zeros_like(u), 1)
    indptr, indices, data = dev.export_csr()
    n = len(u)
    A = np.zeros((n, n))
    for i in range(n):
        A[i, indices[indptr[i]:indptr[i + 1]]] = data[indptr[i]:indptr[i + 1]]
    b = -dev.residual_unconstrained(torch.zeros_like(u)).cpu().numpy()
    bc = dev.bc_dofs.cpu().numpy()
    b[bc] = 0.5
    want = np.linalg.solve(A, b)
    assert np.linalg.norm(u.cpu().numpy() - want) <= 1e-7 * np.linalg.norm(want)
    assert 0 < st['iterations'] <= n
