"""fem_assembly_plan_fill writes the slices' (cell, local node, row lane) pairs to a caller's
buffer, sorted keys (rank * 8 + a) * 64 + lane with the rank that slice_cells gives the cell;
without a buffer the plan is the same, and a buffer without its offsets is refused."""
import numpy as np
import pytest
import torch

from jax_fem_amd import _lib, materials
from jax_fem_amd._lib import check, ptr, stream_ptr
from jax_fem_amd.generate_mesh import Mesh, box_mesh
from jax_fem_amd.problem import Problem

pytestmark = pytest.mark.gpu


class _Law(Problem):
    def get_tensor_map(self):
        return materials.LinearElastic(E=1., nu=0.3)


@pytest.mark.parametrize('n,kind', [((1, 1, 1), 'box'), ((3, 4, 16), 'wedge'), ((5, 6, 7), 'shuffled'), ((30, 1, 1), 'fan')])
def test_pairs(gpu, n, kind):
    m = box_mesh(*n, 1., 1., 1.)
    pts, cells = m.points.copy(), m.cells_dict['hexahedron'].copy()
    rng = np.random.default_rng(3)
    if kind == 'wedge':
        cells[::3, 2], cells[::3, 6] = cells[::3, 3], cells[::3, 7]
    if kind == 'shuffled':
        perm = rng.permutation(len(pts))
        pts, cells = pts[perm], np.argsort(perm)[cells][rng.permutation(len(cells))]
    if kind == 'fan':       # one node of 30 cells
        cells[:, 0] = cells[0, 0]
    dev = _Law(Mesh(pts, cells), vec=3, dim=3).device()
    dm, L, ns, s = dev.dm, dev.L, dev.pat.num_slices, stream_ptr()
    counts, pcounts, err = (dm.empty(k, dtype=torch.int32) for k in (ns, ns, 1))
    check(L.fem_assembly_plan_counts(dev.pref, ptr(dev.inc_ptr), ptr(dev.inc_idx), ptr(counts), ptr(pcounts), ptr(err), s),
          'counts')
    sc_ptr, sp_ptr = dm.scan(counts), dm.scan(pcounts)
    sc, loc = dm.empty(int(sc_ptr[-1]), dtype=torch.int32), dm.empty(dm.C * 64, dtype=torch.int32)
    sc0, loc0 = torch.empty_like(sc), torch.empty_like(loc)
    pairs = torch.full((int(sp_ptr[-1]) + 1,), -7, dtype=torch.int32, device='cuda')
    fill = lambda spp, a, b, c: L.fem_assembly_plan_fill(dev.pref, ptr(dev.inc_ptr), ptr(dev.inc_idx), ptr(sc_ptr), ptr(spp),
                                                         ptr(a), ptr(b), ptr(c), ptr(err), s)
    assert fill(None, sc, pairs, loc) == _lib.FEM_ERR_BAD_ARG
    check(fill(sp_ptr, sc, pairs, loc), 'fill')
    check(fill(None, sc0, None, loc0), 'fill')
    assert int(err) == 0 and torch.equal(sc, sc0) and torch.equal(loc, loc0)
    sc, scp, spp, got = (t.cpu().numpy() for t in (sc, sc_ptr, sp_ptr, pairs))
    inc_ptr, inc_idx = dev.inc_ptr.cpu().numpy(), dev.inc_idx.cpu().numpy()
    sell_row = dev.pat_tensors['sell_row'].cpu().numpy()
    for i in range(ns):
        ends, lists = sc[scp[i]:scp[i] + 8], sc[scp[i] + 8:scp[i + 1]]
        want = []
        for lane in range(64):
            r = sell_row[64 * i + lane]
            if r < 0:
                continue
            first = ends[lane // 8 - 1] if lane >= 8 else 0
            for e in inc_idx[inc_ptr[r]:inc_ptr[r + 1]]:
                rank = first + int(np.searchsorted(lists[first:ends[lane // 8]], e // 8))
                assert lists[rank] == e // 8
                want.append((rank * 8 + e % 8) * 64 + lane)
        assert np.array_equal(got[spp[i]:spp[i + 1]], np.sort(want)), (kind, i)
    assert got[-1] == -7
