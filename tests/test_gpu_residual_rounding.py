"""Rounding of the residuals against sums in extended precision (80 bits).

Hyperelastic: the single-pass assembly's residual rounds no more than the separate one.  Both
form F from the displacement's gradient, J, b or F^-T and J^(-2/3) once each, and the stress
of a small strain is a difference of terms of order 1 that shows those roundings: the errors
(root mean square over the nodes and five fields) are to agree within a tenth."""
import numpy as np
import pytest
import torch

from jax_fem_amd import _lib, materials
from jax_fem_amd.generate_mesh import Mesh, box_mesh, box_mesh_hex27
from jax_fem_amd.problem import Problem

pytestmark = pytest.mark.gpu
LD = np.longdouble


class _Law(Problem):
    law = None

    def get_tensor_map(self):
        return self.law


def _problem(law, n, second=False, vec=3):
    m = (box_mesh_hex27 if second else box_mesh)(*n, 1., 1., 1.)
    x = m.points
    x = x + 0.05 * np.sin(np.pi * x).prod(1, keepdims=True) * np.cos(2. * np.pi * np.roll(x, 1, 1))
    kw = dict(ele_type='HEX27', quadrature_order=4) if second else {}
    p = _Law(Mesh(x, m.cells_dict['hexahedron27' if second else 'hexahedron']), vec=vec, dim=3, **kw)
    p.law = law
    return p


def _field(p, rng, amp):
    x, c = np.asarray(p.fes[0].points), rng.standard_normal((3, 3))
    u = np.stack([c[i, 0] * np.sin(1.5 * x[:, 0]) * x[:, 1] + c[i, 1] * np.cos(2. * x[:, 1]) * x[:, 2] +
                  c[i, 2] * x[:, 2] * x[:, 0] for i in range(3)], 1)
    return amp * (u + 0.01 * rng.standard_normal(u.shape))[:, :p.fes[0].vec]


def _det_inv(J):
    r = [J[..., i, :] for i in range(3)]
    cross = lambda a, b: np.stack([a[..., 1] * b[..., 2] - a[..., 2] * b[..., 1], a[..., 2] * b[..., 0] - a[..., 0] * b[..., 2],
                                   a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]], -1)
    A = np.stack([cross(r[1], r[2]), cross(r[2], r[0]), cross(r[0], r[1])], -1)
    d = (r[0] * A[..., 0]).sum(-1)
    return d, A / d[..., None, None]


def _exact(p, u, stress):
    """Internal forces in 80 bits; stress(G) of (cells, points, vec, 3) displacement gradients."""
    fe = p.fes[0]
    pts, cells = np.asarray(fe.points, dtype=LD), np.asarray(fe.cells)
    dN, w = np.asarray(fe.shape_grads_ref).astype(LD), np.asarray(fe.quad_weights).astype(LD)
    x, ul = pts[cells], u.astype(LD)[cells]
    ul = ul - ul[:, :1]     # (exact; the sums below are good to 19 digits of what they add)
    d, iJ = _det_inv((x[:, None, :, :, None] * dN[None, :, :, None, :]).sum(2))
    g = (dN[None, :, :, :, None] * iJ[:, :, None, :, :]).sum(3)
    G = (ul[:, None, :, :, None] * g[:, :, :, None, :]).sum(2)
    f = ((d * w)[:, :, None, None, None] * stress(G)[:, :, None] * g[:, :, :, None, :]).sum((1, 4))
    out = np.zeros((len(pts), u.shape[1]), LD)
    np.add.at(out, cells, f)
    return out


def _dev(p, u):
    dev = p.device()
    dev.prepare()
    return dev, torch.as_tensor(u, device='cuda').reshape(-1).contiguous()


@pytest.mark.parametrize('amp', [1e-5, 1e-2])
def test_hyperelastic_single_pass_residual(gpu, amp):
    p = _problem(materials.NeoHookean(E=10., nu=0.3), (6, 5, 4))
    err = np.zeros(2)
    for seed in range(5):
        u = _field(p, np.random.default_rng(seed), amp)
        dev, ut = _dev(p, u)
        mu, kappa = (LD(dev.mat_desc.c[i]) for i in range(2))

        def stress(G):
            F = G + np.eye(3, dtype=LD)
            J, Fi = _det_inv(F)
            J, H = J[..., None, None], np.swapaxes(Fi, -1, -2)
            I1 = (F * F).sum((-1, -2), keepdims=True)
            return mu * np.exp(-2 * np.log(J) / 3) * (F - I1 / 3 * H) + kappa * J * (J - 1) * H
        want = _exact(p, u, stress)
        for k, fused in enumerate((True, False)):
            dev.tangent(ut, _lib.FEM_F64, fused=fused, residual=True)
            e = dev.last_residual.cpu().numpy().reshape(-1, 3) - want
            err[k] += float((e * e).sum() / (want * want).sum())
    assert err[0] ** .5 <= 1.1 * err[1] ** .5, err ** .5


@pytest.mark.parametrize('second', [False, True], ids=['hex8', 'hex27'])
@pytest.mark.parametrize('kind', ['poisson', 'elastic', 'simp'])
def test_residual_of_a_translated_body(gpu, kind, second):
    """A strain field of 1e-3 on a translation by a thousand: differences from a cell's first node are
    exact, so the residual keeps its digits, some 50 roundings of its largest entry (1e-14), where
    interpolating the field itself loses six (1e3 / 1e-3)."""
    law = {'poisson': materials.Poisson(k=2.), 'elastic': materials.LinearElastic(E=1., nu=0.3),
           'simp': materials.SIMPElastic(E0=1., Emin=1e-3, nu=0.3, penal=3.)}[kind]
    p = _problem(law, (4, 3, 3) if second else (6, 5, 4), second, 1 if kind == 'poisson' else 3)
    rng = np.random.default_rng(4)
    u = _field(p, rng, 1e-3) + 1e3
    E = np.ones((p.num_cells, p.fes[0].num_quads), LD)
    if kind == 'simp':
        theta = rng.uniform(0.4, 0.6, E.shape)
        p.internal_vars = [torch.as_tensor(theta, device='cuda')]
        E = LD(1e-3) + (1 - LD(1e-3)) * theta.astype(LD) ** 3
    dev, ut = _dev(p, u)
    c = [LD(dev.mat_desc.c[i]) for i in range(2)]

    def stress(G):
        if kind == 'poisson':
            return c[0] * G
        tr = np.trace(G, axis1=-2, axis2=-1)[..., None, None]
        return E[..., None, None] * (c[0] * tr * np.eye(3, dtype=LD) + c[1] * (G + np.swapaxes(G, -1, -2)))
    want = _exact(p, u, stress)
    got = dev.residual_unconstrained(ut).cpu().numpy().reshape(want.shape)
    assert np.abs(got - want).max() <= 1e-14 * np.abs(want).max()
