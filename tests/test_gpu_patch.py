"""Matrix-free patch products (fem_patch_apply, fem_patch_residual) and the solves
that run on them, against the assembled matrix and the two-pass residual, at the edges of the patches (one cell, 127 / 128 / 129 HEX8 and 27 / 28 / 29 HEX27 cells),
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
from jax_fem_amd.generate_mesh import Mesh, box_mesh, box_mesh_hex27
from jax_fem_amd.problem import Problem
from jax_fem_amd.solver import linear_config, solver
from problems import isclose

pytestmark = pytest.mark.gpu


def _mesh(n, shuffle=False, second=False):
    m = (box_mesh_hex27 if second else box_mesh)(*n, 1., n[1] / n[0], n[2] / n[0])
    pts, cells = m.points.copy(), m.cells_dict['hexahedron27' if second else 'hexahedron']
    rng = np.random.default_rng(3)
    pts += (0.05 if second else 0.1) / n[0] * rng.uniform(-1., 1., pts.shape)
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


def _problem(kind, n, shuffle=False, second=False):
    clamp = lambda v: [[lambda x: isclose(x[0], 0.)] * v, list(range(v)), [lambda x: 0.] * v]
    vec = 1 if kind == 'poisson' else 3
    kw = dict(ele_type='HEX27', quadrature_order=4) if second else {}
    p = _Law(_mesh(n, shuffle, second), vec=vec, dim=3, dirichlet_bc_info=clamp(vec), **kw)
    p.law = {'poisson': materials.Poisson(k=2.5), 'elastic': materials.LinearElastic(E=70e3, nu=0.3),
             'simp': materials.SIMPElastic(E0=1., Emin=1e-3, nu=0.3, penal=3.),
             'neo': materials.NeoHookean(E=10., nu=0.3)}[kind]
    if kind == 'simp':
        theta = 0.3 + torch.rand((p.num_cells, p.fes[0].num_quads), dtype=torch.float64, device='cuda',
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
@pytest.mark.parametrize('n,shuffle,second', [
    ((1, 1, 1), False, False), ((127, 1, 1), False, False), ((4, 4, 8), False, False), ((43, 3, 1), False, False),
    ((9, 7, 5), True, False), ((1, 1, 1), False, True), ((9, 3, 1), False, True), ((7, 2, 2), False, True),
    ((29, 1, 1), False, True), ((5, 4, 3), True, True)],
    ids=['1', '127', '128', '129', 'shuffled', 'hex27_1', 'hex27_27', 'hex27_28', 'hex27_29', 'hex27_shuffled'])
def test_patch_product_and_residual_match_the_assembled(gpu, kind, n, shuffle, second):
    p = _problem(kind, n, shuffle, second)
    dev = p.device()
    dev.prepare()
    u = _u(p)
    dev.tangent(u, _lib.FEM_F64, fused=False)
    v = _u(p, 1.)
    ref = dev.spmv(v)
    modulus = None
    if kind == 'simp':
        modulus = torch.empty(p.num_cells * p.fes[0].num_quads, dtype=torch.float64, device='cuda')
        check(dev.L.fem_patch_modulus(dev.dm.ref, dev.mref, ptr(modulus), stream_ptr()), 'fem_patch_modulus')
    for mod in ({None, modulus} if kind != 'neo' or not second else ()):   # no HEX27 hyperelastic tangent
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
    op = dev.patch_operator(dev.mat_desc)
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


OPTIONS = [{'jax_solver': {'precision': 'fp64'}}, {'jax_solver': {'precision': 'mixed'}},
           {'amgx_solver': {'precision': 'fp64'}}, {'amgx_solver': {'precision': 'mixed'}},
           {'amgx_solver': {'precision': 'mixed', 'setup_reuse': 2}}]
OPTION_IDS = ['pcg64', 'pcg_mixed', 'amg64', 'amg_mixed', 'amg_reuse']


@pytest.mark.parametrize('kind', ['simp', 'neo'])
@pytest.mark.parametrize('options', OPTIONS, ids=OPTION_IDS)
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
        monkeypatch.setattr(dev, 'patch_min_cells', lambda storage: min_cells)
        dev.drop_amg_hierarchy()
        sols.append(solver(p, opts)[0].clone())
        storage = _lib.FEM_F32 if options[key].get('precision') == 'mixed' else _lib.FEM_F64
        free_of_matrix = min_cells == 0 and not (kind == 'neo' and storage == _lib.FEM_F32)
        assert (dev.fine_for(storage) is not None) == free_of_matrix
    assert torch.linalg.norm(sols[1] - sols[0]) <= 1e-9 * torch.linalg.norm(sols[0])
    # a second solve gives the same bits
    dev.drop_amg_hierarchy()
    assert torch.equal(solver(p, opts)[0], sols[1])


@pytest.mark.parametrize('options', OPTIONS, ids=OPTION_IDS)
def test_hex27_matrix_free_solves_meet_their_tolerance(gpu, options, monkeypatch):
    # the solver stops at |b - A x| <= rtol |b| on its own operator; the assembled FP64 matrix
    # differs from that by rounding, some 1e-16 |A| |x| <= 1e-12 |b| here (|A| |x| <= 1e4 |b|)
    p = _problem('simp', (6, 5, 4), second=True)
    key = next(iter(options))
    rtol = 1e-10
    dev = p.device()
    dev.prepare()
    monkeypatch.setattr(dev, 'patch_min_cells', lambda storage: 0)
    u0 = torch.zeros(dev.n, dtype=torch.float64, device='cuda')
    b = _u(p, 1.)
    b[dev.bc_dofs_long] = 0.
    cfg = linear_config({key: dict(options[key], tol=rtol, atol=0.)})
    dev.tangent(u0, cfg['precision_code'])
    assert dev.fine_for(_lib.FEM_F32 if options[key]['precision'] == 'mixed' else _lib.FEM_F64) is not None
    x, info = dev.solve(u0, b, torch.zeros_like(b), cfg)
    assert info.status == _lib.FEM_OK and info.iterations > 1
    dev.tangent(u0, _lib.FEM_F64)
    assert torch.linalg.norm(b - dev.spmv(x)) <= 1.1 * rtol * torch.linalg.norm(b)
