"""Rows longer than a box mesh has: a fan of hexahedra around one edge, stacked along it.

One-workgroup Jacobi-PCG (k_pcg_one): rows of 75 blocks, of which 32 are held and the rest read
where they are, in the first slices (matrix in registers) and in the last (matrix in LDS); and
iteration limits inside a batch.  Single-pass assembly: rows of 30 blocks, and of 34, which it
leaves to the two-pass path.

Tolerances: solves meet rtol 1e-11 on the residual; the condition number is below 1e4, so they
agree with dense ones to 1e-7 (truncated ones, a few steps of one recursion in other orders of
summation, to 1e-11).  Assembly: another order of the same FP64 sums, 1e-13 of the largest entry."""
import numpy as np
import pytest
import torch

from jax_fem_amd import _lib, materials
from jax_fem_amd.generate_mesh import Mesh
from jax_fem_amd.problem import Problem
from jax_fem_amd.solver import linear_config
from problems import isclose

pytestmark = pytest.mark.gpu


class _Law(Problem):
    law = materials.Poisson(k=2.)

    def get_tensor_map(self):
        return self.law


def _fan(k, layers, axis):
    """k cells around the z axis, `layers` of them; the axis' nodes numbered first, last or where they fall."""
    t = 2. * np.pi * np.arange(k) / k
    plane = np.vstack([[[0., 0.]], np.c_[np.cos(t), np.sin(t)], 1.4 * np.c_[np.cos(t + np.pi / k), np.sin(t + np.pi / k)]])
    P = len(plane)
    pts = np.vstack([np.c_[plane, np.full(P, z)] for z in np.linspace(0., 1., layers + 1)])
    i = np.arange(k)
    quad = np.c_[0 * i, 1 + i, 1 + k + i, 1 + (i + 1) % k]
    cells = np.vstack([np.hstack([quad + P * l, quad + P * (l + 1)]) for l in range(layers)])
    on = np.arange(len(pts)) % P == 0
    order = np.argsort({'first': ~on, 'last': on, 'natural': 0 * on}[axis], kind='stable')
    return Mesh(pts[order], np.argsort(order)[cells])


def _dense(dev):
    indptr, indices, data = dev.export_csr()
    A = np.zeros((dev.n, dev.n))
    A[np.repeat(np.arange(dev.n), np.diff(indptr)), indices] = data
    return A


def _scalar(monkeypatch, axis, k=12, layers=43):
    L = _lib.lib()
    natural = L.fem_sell_order       # rows in the order of the nodes, so that the axis' slices can be chosen
    monkeypatch.setattr(L, 'fem_sell_order', lambda n, sort, *a: natural(n, 0, *a))
    p = _Law(_fan(k, layers, axis), vec=1, dim=3,
             dirichlet_bc_info=[[lambda x: isclose(x[2], 0.)], [0], [lambda x: 0.]])
    dev = p.device()
    dev.prepare()
    b = torch.randn(dev.n, dtype=torch.float64, device='cuda', generator=torch.Generator(device='cuda').manual_seed(4))
    b[dev.bc_dofs_long] = 0.
    slots = np.diff(dev.pat_tensors['slice_ptr'].cpu().numpy()) // 64
    assert dev.pat.num_slices == 18 and dev.pat.sell_blocks <= 18 * 64 * 32     # what the one-workgroup form takes
    assert slots[0 if axis == 'first' else 17] == 3 * (1 + 2 * k)
    return dev, b


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('axis', ['first', 'last'])
def test_one_workgroup_solve(gpu, axis, precision, monkeypatch):
    dev, b = _scalar(monkeypatch, axis)
    cfg = linear_config({'jax_solver': dict(precision=precision, tol=1e-11, atol=0.)})
    u = torch.zeros_like(b)
    dev.tangent(u, cfg['precision_code'])
    x, info = dev.solve(u, b, torch.zeros_like(b), cfg)
    two, launched = dev.solve(u, b, torch.zeros_like(b), dict(cfg, timing=True))    # the two-launch form
    assert info.status == launched.status == _lib.FEM_OK and abs(info.iterations - launched.iterations) <= 2 + 0.03 * info.iterations
    dev.tangent(u, _lib.FEM_F64)
    want = np.linalg.solve(_dense(dev), b.cpu().numpy())
    for got in (x, two):
        assert np.linalg.norm(got.cpu().numpy() - want) <= 1e-7 * np.linalg.norm(want)


@pytest.mark.parametrize('limit', [1, 5, 16, 21])
def test_limit_inside_a_batch(gpu, limit, monkeypatch):
    dev, b = _scalar(monkeypatch, 'last')
    cfg = linear_config({'jax_solver': dict(precision='fp64', tol=1e-11, atol=0., maxiter=limit, check_every=16)})
    u = torch.zeros_like(b)
    dev.tangent(u, _lib.FEM_F64)
    x, info = dev.solve(u, b, torch.zeros_like(b), cfg)
    assert info.status == _lib.FEM_ERR_NOT_CONVERGED and info.iterations == limit
    A, r = _dense(dev), b.cpu().numpy()
    want, d = np.zeros(dev.n), 1. / np.diag(A)
    z = d * r
    p, rz = z, r @ z
    for _ in range(limit):
        q = A @ p
        alpha = rz / (p @ q)
        want, r = want + alpha * p, r - alpha * q
        z = d * r
        rz, old = r @ z, rz
        p = z + rz / old * p
    assert np.linalg.norm(x.cpu().numpy() - want) <= 1e-11 * np.linalg.norm(want)
    assert abs(info.res_norm - np.linalg.norm(r)) <= 1e-11 * np.linalg.norm(b.cpu().numpy())


@pytest.mark.parametrize('law', ['poisson', 'elastic', 'neo'])
@pytest.mark.parametrize('k', [7, 8])
def test_assembly(gpu, k, law):
    vec = 1 if law == 'poisson' else 3
    p = _Law(_fan(k, 1, 'natural'), vec=vec, dim=3)
    p.law = {'poisson': materials.Poisson(k=2.), 'elastic': materials.LinearElastic(E=70e3, nu=0.3),
             'neo': materials.NeoHookean(E=10., nu=0.3)}[law]
    dev = p.device()
    dev.prepare()
    u = 0.02 * torch.randn(dev.n, dtype=torch.float64, device='cuda', generator=torch.Generator(device='cuda').manual_seed(4))
    assert dev.fused_applies(_lib.FEM_F64) == (2 * (1 + 2 * k) <= 32)
    for precision, tol in ((_lib.FEM_F64, 1e-13), (_lib.FEM_F32, 1e-6)):
        dev.tangent(u, precision, residual=True)
        got = [t.double().clone() for t in (dev.current[2], dev.current[3], dev.last_residual)]
        dev.tangent(u, precision, residual=True, fused=False)
        for a, b, t in zip(got, (dev.current[2], dev.current[3], dev.last_residual), (tol, tol, 1e-12)):
            assert float((a - b.double()).abs().max()) <= t * float(b.abs().max())
