"""Single-pass assembly in groups of eight rows, at the sizes where groups, chunks and
slices end, on node numbers without locality, and with cells that name a node twice
(collapsed to wedges): every law and both storage forms against the two-pass path.

Tolerances: both sides sum the same few hundred FP64 products per entry in another
order, so they agree to 1e-13 of the largest entry (1e-12 for the residual, whose terms
cancel); the FP32 form rounds the same FP64 sums once."""
import numpy as np
import pytest
import torch

from jax_fem_amd import _lib, materials as M
from jax_fem_amd.generate_mesh import Mesh, box_mesh
from jax_fem_amd.problem import Problem
from problems import Plasticity, isclose

pytestmark = pytest.mark.gpu


class _Law(Problem):
    law = None

    def get_tensor_map(self):
        return self.law


LAWS = {'poisson': M.Poisson(k=2.5), 'elastic': M.LinearElastic(E=70e3, nu=0.3),
        'simp': M.SIMPElastic(E0=1., Emin=1e-3, nu=0.3, penal=3.), 'simp_frac': M.SIMPElastic(penal=2.5),
        'neo': M.NeoHookean(E=10., nu=0.3), 'j2': None}


def _mesh(n, order):
    m = box_mesh(*n, 1., n[1] / n[0], n[2] / n[0])
    pts, cells = m.points.copy(), m.cells_dict['hexahedron'].copy()
    rng = np.random.default_rng(3)
    pts += 0.05 / n[0] * rng.uniform(-1., 1., pts.shape)
    if order == 'wedge':   # the quads 0-1-2-3 and 4-5-6-7 become triangles
        c = np.arange(0, len(cells), 3)
        cells[c, 2], cells[c, 6] = cells[c, 3], cells[c, 7]
    if order == 'shuffled':
        perm = rng.permutation(len(pts))
        pts, cells = pts[perm], np.argsort(perm)[cells][rng.permutation(len(cells))]
    return Mesh(pts, cells)


@pytest.mark.parametrize('law', list(LAWS))
@pytest.mark.parametrize('n,order', [((1, 1, 1), 'natural'), ((1, 1, 7), 'natural'), ((1, 2, 8), 'wedge'),
                                     ((2, 3, 9), 'shuffled'), ((3, 4, 16), 'wedge'), ((2, 2, 70), 'natural')])
def test_groups_match_two_pass(gpu, law, n, order):
    mesh, rng = _mesh(n, order), np.random.default_rng(5)
    vec = 1 if law == 'poisson' else 3
    cls = Plasticity if law == 'j2' else _Law
    p = cls(mesh, vec=vec, dim=3, dirichlet_bc_info=[[lambda x: isclose(x[0], 0.)] * vec, list(range(vec)),
                                                     [lambda x: 0.] * vec])
    C, Q = p.num_cells, p.fes[0].num_quads
    if law == 'j2':
        sym = lambda a: torch.as_tensor(0.5 * (a + np.swapaxes(a, -1, -2)))
        p.internal_vars = [sym(150. * rng.standard_normal((C, Q, 3, 3))), sym(2e-3 * rng.standard_normal((C, Q, 3, 3)))]
    else:
        p.law = LAWS[law]
        if law.startswith('simp'):
            p.internal_vars = [torch.as_tensor(rng.uniform(0.2, 1., (C, Q)))]
    u = torch.as_tensor((2e-3 if law == 'j2' else 2e-2) / n[0] * rng.standard_normal(p.fes[0].num_total_dofs),
                        device='cuda')
    dev = p.device()
    dev.prepare()
    assert dev.fused_applies(_lib.FEM_F64)
    for precision, tol in ((_lib.FEM_F64, 1e-13), (_lib.FEM_F32, 1e-6)):
        out = []
        for fused in (True, False):
            dev.tangent(u, precision, fused=fused, residual=True)
            out.append([t.double().clone() for t in (dev.current[2], dev.current[3], dev.last_residual)])
        dev.tangent(u, precision)     # the kernel without the residual
        out[0].append(dev.current[2].double().clone())
        for a, b, t in zip(out[0], out[1] + out[1][:1], (tol, tol, 1e-12, tol)):
            assert float(b.abs().max()) > 0.
            assert float((a - b).abs().max()) <= t * float(b.abs().max()), (precision, t)
