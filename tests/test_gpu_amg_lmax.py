"""fem_amg_lmax without a SELL pattern estimates on the block CSR matrix, whatever sell_f32
and sell_vals are: the storage code of a matrix-free operator there neither dereferences
sell_vals nor changes the estimate (bit for bit: the same kernels on the same matrix)."""
import ctypes as C

import pytest
import torch

from jax_fem_amd import _lib
from jax_fem_amd._lib import ptr, stream_ptr
from jax_fem_amd.amg import POWER_STEPS, Bcsr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('f32', [False, True], ids=['fp64', 'fp32'])
def test_storage_code_without_a_pattern(gpu, f32):
    L, n, dev = _lib.load(), 200, torch.device('cuda')
    # tridiagonal, 1 x 1 blocks
    ci = [[c for c in (r - 1, r, r + 1) if 0 <= c < n] for r in range(n)]
    rp = torch.tensor([0] + [len(c) for c in ci], device=dev).cumsum(0).to(torch.int32)
    cols = torch.tensor(sum(ci, []), dtype=torch.int32, device=dev)
    rows = torch.arange(n, device=dev).repeat_interleave(torch.diff(rp.long()))
    vals = torch.where(cols.long() == rows, 4., -1.).to(torch.float32 if f32 else torch.float64)
    s = Bcsr(n, n, 1, 1, rp, cols, vals).struct()
    dinv = torch.full((n,), .25, dtype=torch.float64, device=dev)
    ws = torch.empty(int(L.fem_amg_lmax_ws_bytes(n)), dtype=torch.uint8, device=dev)
    got = []
    for code in (0, 3):
        lam, lam_dev = C.c_double(0.), torch.zeros(1, dtype=torch.float64, device=dev)
        assert L.fem_amg_lmax(C.byref(s), None, None, code, ptr(dinv), POWER_STEPS, C.byref(lam), ptr(ws),
                              stream_ptr()) == _lib.FEM_OK
        assert L.fem_amg_lmax_async(C.byref(s), None, None, code, ptr(dinv), POWER_STEPS, ptr(lam_dev), ptr(ws),
                                    stream_ptr()) == _lib.FEM_OK
        got += [lam.value, float(lam_dev)]
    assert len(set(got)) == 1 and 1. < got[0] < 1.5, got
