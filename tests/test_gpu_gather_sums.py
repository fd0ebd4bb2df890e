"""Row sums of the difference form (fem_gather_matrix): FP64 sums rounded once, also where the
cell tangents are FP32.

Input: cell tangents of whole numbers below 2^20, so that every block's sum (at most 8 cells)
is exact in FP32 while a row's sum of up to 27 or 125 blocks is exact in FP64 only: the stored
row sum is that sum's nearest FP32 number, bit for bit, in any order of summation."""
import numpy as np
import pytest
import torch

from jax_fem_amd import _lib, materials as M
from jax_fem_amd._lib import check, ptr, stream_ptr
from jax_fem_amd.generate_mesh import Mesh, box_mesh, box_mesh_hex27
from jax_fem_amd.problem import Problem

pytestmark = pytest.mark.gpu


class _Law(Problem):
    def get_tensor_map(self):
        return M.LinearElastic(E=1., nu=0.3)


@pytest.mark.parametrize('ele,precision', [('HEX8', 'f32'), ('HEX8', 'f64'), ('HEX27', 'f32'), ('HEX27', 'f64')])
def test_row_sums_are_rounded_once(gpu, ele, precision):
    second = ele == 'HEX27'
    m = (box_mesh_hex27 if second else box_mesh)(*((2, 3, 2) if second else (5, 4, 6)), 1., 1., 1.)
    cells = m.cells_dict['hexahedron27' if second else 'hexahedron']
    p = _Law(Mesh(m.points, cells), vec=3, dim=3, ele_type=ele, **(dict(quadrature_order=4) if second else {}))
    dev = p.device()
    dev.prepare()
    C, N = cells.shape
    Ke = np.random.default_rng(3).integers(-2**20, 2**20, (C, N, N, 3, 3)).astype(np.float64)
    rows = np.zeros((len(m.points), 3, 3))
    np.add.at(rows, cells.reshape(-1), Ke.sum(2).reshape(-1, 3, 3))
    f32 = precision == 'f32'
    K = torch.as_tensor(Ke, dtype=torch.float32 if f32 else torch.float64, device='cuda')
    vals = torch.zeros((int(dev.pat.sell_blocks) * 9,), dtype=torch.float32, device='cuda')
    check(dev.L.fem_gather_matrix(dev.pref, _lib.FEM_F32 if f32 else _lib.FEM_F64, ptr(K), _lib.FEM_F32,
                                  _lib.FEM_FORM_DIFFERENCE, ptr(vals), None, stream_ptr()), 'gather')
    v = vals.cpu().numpy()
    ds, sell_row, slice_ptr = (dev.pat_tensors[k].cpu().numpy() for k in ('diag_slot', 'sell_row', 'slice_ptr'))
    got = np.zeros((len(m.points), 3, 3), dtype=np.float32)
    for lane, r in enumerate(sell_row):
        if r >= 0:
            s, l = divmod(lane, 64)
            got[r] = v[9 * slice_ptr[s]:9 * slice_ptr[s + 1]].reshape(-1, 3, 3, 64)[ds[r], ..., l]
    assert np.array_equal(got, rows.astype(np.float32))
