"""Matrix-free patch products (fem_patch_apply, fem_patch_residual) and the solves
that run on them, against the assembled matrix, the two-pass residual and the
oracle, at the edges of the patches (one cell, 127 / 128 / 129 cells, odd boxes),
on meshes whose cells are not consecutive in space, and with FP32 vectors.

Tolerances: both sides sum at most a few hundred FP64 products per entry, so
they agree to 1e-13 of the largest entry; solves to rtol 1e-12 agree to 1e-9
(condition numbers up to 1e5 here)."""
import ctypes as C

import numpy as np
import pytest
import torch

from jax_fem_amd import _lib, materials
from jax_fem_amd._lib import check, ptr, stream_ptr
from jax_fem_amd.generate_mesh import Mesh, box_mesh
from jax_fem_amd.problem import Problem
from jax_fem_amd.solver import solver
from problems import isclose

pytestmark = pytest.mark.gpu


def _mesh(n, shuffle=False):
    m = box_mesh(*n, 1., n[1] / n[0], n[2] / n[0])
    pts, cells = m.points.copy(), m.cells_dict['hexahedron']
    rng = np.random.default_rng(3)
    pts += 0.1 / n[0] * rng.uniform(-1., 1., pts.shape)
    pts[isclose(m.points[:, 0], 0.)] = m.points[isclose(m.points[:, 0], 0.)]
    if shuffle:   # node and cell numbers without locality
        perm = rng.permutation(len(pts))
        inv = np.argsort(perm)
        pts, cells = pts[perm], inv[cells][rng.permutation(len(cells))]
    return Mesh(pts, cells)


class _Law(Problem):
    law = None

    def get_tensor_map(self):
        return self.law

    def set_params(self, theta):
        self.internal_vars = [theta]


def _problem(kind, n, shuffle=False):
    clamp = lambda v: [[lambda x: isclose(x[0], 0.)] * v, list(range(v)), [lambda x: 0.] * v]
    vec = 1 if kind == 'poisson' else 3
    p = _Law(_mesh(n, shuffle), vec=vec, dim=3, dirichlet_bc_info=clamp(vec))
    p.law = {'poisson': materials.Poisson(k=2.5), 'elastic': materials.LinearElastic(E=70e3, nu=0.3),
             'simp': materials.SIMPElastic(E0=1., Emin=1e-3, nu=0.3, penal=3.),
             'neo': materials.NeoHookean(E=10., nu=0.3)}[kind]
    if kind == 'simp':
        theta = 0.3 + torch.rand((p.num_cells, 8), dtype=torch.float64, device='cuda',
                                 generator=torch.Generator(device='cuda').manual_seed(1))
        p.set_params(theta)
    return p


def _u(p, scale=0.02):
    """A rough field of the given size in cells (all cells are about cubes)."""
    g = torch.Generator(device='cuda').manual_seed(5)
    x = np.asarray(p.fes[0].points)[np.asarray(p.fes[0].cells)[0, :2], :]
    return scale * float(np.linalg.norm(x[1] - x[0])) * torch.randn(p.fes[0].num_total_dofs, dtype=torch.float64,
                                                                    device='cuda', generator=g)


@pytest.mark.parametrize('kind', ['poisson', 'elastic', 'simp', 'neo'])
@pytest.mark.parametrize('n,shuffle', [((1, 1, 1), False), ((127, 1, 1), False), ((4, 4, 8), False),
                                       ((43, 3, 1), False), ((9, 7, 5), True)],
                         ids=['1cell', '127', '128', '129', 'shuffled'])
def test_patch_product_and_residual_match_the_assembled(gpu, kind, n, shuffle):
    p = _problem(kind, n, shuffle)
    dev = p.device()
    dev.prepare()
    u = _u(p)
    dev.tangent(u, _lib.FEM_F64, fused=False)
    v = _u(p, 1.)
    ref = dev.spmv(v)
    modulus = None
    if kind == 'simp':
        modulus = torch.empty(p.num_cells * 8, dtype=torch.float64, device='cuda')
        check(dev.L.fem_patch_modulus(dev.dm.ref, dev.mref, ptr(modulus), stream_ptr()), 'fem_patch_modulus')
    for mod in {None, modulus}:
        op = dev.patch_operator(dev.mat_desc, u, mod)
        y = torch.empty_like(v)
        check(dev.L.fem_patch_apply(C.byref(op), ptr(v), ptr(y), stream_ptr()), 'fem_patch_apply')
        free = dev.bc_mask == 0
        assert float((y - ref).abs()[free].max()) <= 1e-13 * float(ref[free].abs().max())
        assert torch.equal(y[~free], v[~free])
    # the residual: patches against the per-cell vectors and their nodal gather
    cell = dev.cell_buffer()
    check(dev.L.fem_cell_residual(dev.dm.ref, dev.mref, ptr(u), ptr(cell), stream_ptr()), 'fem_cell_residual')
    base = _u(p, 3.)
    want, got = torch.empty_like(u), torch.empty_like(u)
    check(dev.L.fem_gather_nodal(dev.dm.Nn, dev.V, ptr(dev.inc_ptr), ptr(dev.inc_idx), ptr(cell), ptr(base), ptr(want),
                                 stream_ptr()), 'fem_gather_nodal')
    check(dev.L.fem_patch_residual(C.byref(op), ptr(u), ptr(base), ptr(got), stream_ptr()), 'fem_patch_residual')
    assert float((got - want).abs().max()) <= 1e-13 * float(want.abs().max())


def test_patch_residual_of_an_inverted_element_is_nan(gpu):
    # J < 0: J^(-2/3) has no value; the products give NaN as the assembled law does
    p = _problem('neo', (2, 2, 2))
    dev = p.device()
    dev.prepare()
    u = -2.2 * torch.as_tensor(p.fes[0].points, device='cuda').reshape(-1)
    op = dev.patch_operator(dev.mat_desc, u)
    y = torch.empty_like(u)
    check(dev.L.fem_patch_apply(C.byref(op), ptr(u), ptr(y), stream_ptr()), 'fem_patch_apply')
    free = dev.bc_mask == 0
    assert bool(torch.isnan(y[free]).all())
    assert bool(torch.isnan(dev.residual_unconstrained(u)).any())


@pytest.mark.parametrize('kind', ['simp', 'neo'])
@pytest.mark.parametrize('options', [{'jax_solver': {'precision': 'fp64'}}, {'jax_solver': {'precision': 'mixed'}},
                                     {'amgx_solver': {'precision': 'fp64'}}, {'amgx_solver': {'precision': 'mixed'}},
                                     {'amgx_solver': {'precision': 'mixed', 'setup_reuse': 2}}],
                         ids=['pcg64', 'pcg_mixed', 'amg64', 'amg_mixed', 'amg_reuse'])
def test_matrix_free_solves_match_the_matrix_solves(gpu, kind, options, monkeypatch):
    p = _problem(kind, (14, 9, 8))
    key = next(iter(options))
    opts = {key: dict(options[key], tol=1e-12 if key == 'amgx_solver' else 1e-11, atol=0.), 'tol': 1e-10,
            'rel_tol': 1e-13}
    p.fes[0].update_Dirichlet_boundary_conditions(
        [[lambda x: isclose(x[0], 0.)] * 3 + [lambda x: x[0] > 0.97], [0, 1, 2, 1],
         [lambda x: 0.] * 3 + [lambda x: 0.02]])
    dev = p.device()
    sols = []
    for min_cells in (1 << 30, 0):
        monkeypatch.setattr(dev, 'PATCH_MIN_CELLS', {_lib.FEM_F64: min_cells, _lib.FEM_F32: min_cells},
                            raising=False)
        dev.drop_amg_hierarchy()
        sols.append(solver(p, opts)[0].clone())
        storage = _lib.FEM_F32 if options[key].get('precision') == 'mixed' else _lib.FEM_F64
        free_of_matrix = min_cells == 0 and not (kind == 'neo' and storage == _lib.FEM_F32)
        assert (dev.fine_for(storage) is not None) == free_of_matrix
    assert torch.linalg.norm(sols[1] - sols[0]) <= 1e-9 * torch.linalg.norm(sols[0])
    # a second solve gives the same bits
    dev.drop_amg_hierarchy()
    assert torch.equal(solver(p, opts)[0], sols[1])
