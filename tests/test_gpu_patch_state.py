"""A solve on the matrix-free operator solves the tangent that was assembled, whatever the
program does to its own tensors after that, and whichever tangent an AMG hierarchy was set
up on: the residual on the assembled FP64 matrix meets the solver's own tolerance (1.1 times
it: the two operators differ by rounding)."""
import pytest
import torch

from jax_fem_amd import _lib, materials
from jax_fem_amd.generate_mesh import Mesh, box_mesh
from jax_fem_amd.problem import Problem
from jax_fem_amd.solver import linear_config
from problems import isclose

pytestmark = pytest.mark.gpu
RTOL = 1e-9


class _Law(Problem):
    law = None

    def get_tensor_map(self):
        return self.law


def _setup(law, options, monkeypatch, param):
    m = box_mesh(9, 8, 7, 1., 1., 1.)
    p = _Law(Mesh(m.points, m.cells_dict['hexahedron']), vec=3, dim=3,
             dirichlet_bc_info=[[lambda x: isclose(x[0], 0.)] * 3, [0, 1, 2], [lambda x: 0.] * 3])
    p.law = law
    gen = torch.Generator(device='cuda').manual_seed(1)
    rand = lambda *shape: torch.rand(shape, dtype=torch.float64, device='cuda', generator=gen)
    if param:
        p.internal_vars = [0.5 + rand(p.num_cells, p.fes[0].num_quads)]
    dev = p.device()
    dev.prepare()
    monkeypatch.setattr(dev, 'patch_min_cells', lambda storage: 0)
    cfg = linear_config({next(iter(options)): dict(options[next(iter(options))], tol=RTOL, atol=0.)})
    b = rand(dev.n) - 0.5
    b[dev.bc_dofs_long] = 0.
    return p, dev, cfg, b, 0.02 * (rand(dev.n) - 0.5)


def _solved(dev, cfg, u, b):
    """|b - A x| of a solve on the matrix assembled beside the operator."""
    x, info = dev.solve(u, b, torch.zeros_like(b), cfg)
    assert info.status == _lib.FEM_OK and info.iterations > 1
    return float(torch.linalg.norm(b - dev.spmv(x)))


@pytest.mark.parametrize('options', [{'jax_solver': {'precision': 'fp64'}}, {'amgx_solver': {'precision': 'fp64'}}],
                         ids=['pcg', 'amg'])
@pytest.mark.parametrize('kind', ['neo', 'simp'])
def test_parameters_edited_after_the_tangent(gpu, kind, options, monkeypatch):
    law = materials.NeoHookean(E=10., nu=0.3, param=True) if kind == 'neo' else \
        materials.SIMPElastic(E0=1., Emin=1e-3, nu=0.3, penal=3.)
    p, dev, cfg, b, u = _setup(law, options, monkeypatch, True)
    dev.tangent(u, cfg['precision_code'])
    assert dev.fine_for(_lib.FEM_F64) is not None
    p.internal_vars[0].mul_(3.)
    u_was = u.clone()
    u.mul_(-1.)
    assert _solved(dev, cfg, u_was, b) <= 1.1 * RTOL * float(torch.linalg.norm(b))


@pytest.mark.parametrize('kind', ['neo', 'simp'])
def test_reused_hierarchy_follows_the_tangent(gpu, kind, monkeypatch):
    law = materials.NeoHookean(E=10., nu=0.3) if kind == 'neo' else materials.SIMPElastic(E0=1., Emin=1e-3, nu=0.3, penal=3.)
    p, dev, cfg, b, u = _setup(law, {'amgx_solver': {'precision': 'fp64', 'setup_reuse': 2}}, monkeypatch, kind == 'simp')
    for step in range(4):
        if kind == 'simp':
            p.internal_vars = [p.internal_vars[0] * 0.8]
            dev.prepare()
        v = (1. + step) * u
        dev.tangent(v, cfg['precision_code'])
        assert dev.fine_for(_lib.FEM_F64) is not None
        err = _solved(dev, cfg, v, b)
        assert err <= 1.1 * RTOL * float(torch.linalg.norm(b)), (step, err)
        assert dev._amg_uses == (0, 1, 2, 0)[step]
