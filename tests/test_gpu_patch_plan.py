"""Which problems hold the plan of the matrix-free products: those whose law a patch kernel
runs, from the start when the program names the law, else once it is recognised; never J2,
tabulated laws and weak forms, which would build it for nothing."""
import pytest
import torch

from problems import box, energy_kernel_torch, svk_torch

from jax_fem_amd import _lib, materials
from jax_fem_amd.problem import Problem

pytestmark = pytest.mark.gpu


class _Law(Problem):
    law = None

    def get_tensor_map(self):
        return self.law


class _Form(Problem):
    def get_universal_kernel(self):
        return energy_kernel_torch(torch.as_tensor(self.fes[0].shape_vals, device='cuda'))


def _isotropic(g):
    e = 0.5 * (g + g.T)
    return 0.6 * torch.trace(e) * torch.eye(3, dtype=g.dtype) + 0.8 * e


LAWS = {'elastic': (materials.LinearElastic(E=1., nu=0.3), True, True), 'neo': (materials.NeoHookean(E=1., nu=0.3), True, True),
        'poisson': (materials.Poisson(k=2.), True, True), 'callable': (_isotropic, False, True),
        'svk': (svk_torch, False, False), 'j2': (materials.J2Plastic(E=70e3, nu=0.3, sig0=250.), False, False),
        'form': (None, False, False)}


@pytest.mark.parametrize('kind', list(LAWS))
def test_who_holds_a_plan(gpu, kind):
    law, at_start, in_use = LAWS[kind]
    vec = 1 if kind in ('poisson', 'form') else 3
    p = (_Form if kind == 'form' else _Law)(box(4, 3, 3), vec=vec, dim=3)
    p.law = law
    if kind == 'j2':
        shape = (p.num_cells, p.fes[0].num_quads, 3, 3)
        p.internal_vars = [torch.zeros(shape, dtype=torch.float64, device='cuda') for _ in range(2)]
    dev = p.device()
    held = lambda: bool(dev.dm._patch) and 'patch_part' in dev.buffers
    assert held() == at_start
    u = torch.full((dev.n,), 1e-3, dtype=torch.float64, device='cuda') * torch.arange(dev.n, device='cuda').sin()
    dev.prepare()
    dev.tangent(u, _lib.FEM_F64, residual=True)
    assert bool(torch.isfinite(dev.residual_unconstrained(u)).all())
    assert held() == in_use and dev.patch_law == in_use
    assert in_use or dev.dm._patch is None
