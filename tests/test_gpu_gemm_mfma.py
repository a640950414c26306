"""The 256-row GEMM kernel (csrc/gemm_mfma.hip) in each of its forms: whole and
padded widths, tiles split along K, f32 planes.  The calls are those of
gemm_cases.py, whose kernels test_gemm_plan.py asserts.

Bars: compare() of tests/_gpu.py, against the f64 oracle and the oracle with
the kernels' storage roundings.
"""
import numpy as np
import pytest
import torch

from _common import rounded, small_case
from _gpu import compare, layer_from_tensors, to_device
from gemm_cases import EXPERTS, ONE_EXPERT
import nomas_moe as nm
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


def check(rows, D, E, k, H, dtype, seed):
    print(f"rows={rows} D={D} E={E} k={k} H={H} {dtype}", flush=True)
    t, x = small_case(rows, D, E, k, H, seed, router_std=0.3)
    layer = layer_from_tensors(t, dtype, D, H, E, k)
    rt, rx = rounded(t, x, dtype)
    p, dn = nm.workloads.oracle_params(rt, E)
    xd = to_device(x, dtype)
    # every tile row offset near the edges of the tiles, all along the call
    sel = np.unique(np.r_[np.arange(0, rows, 113), np.arange(250, 262), np.arange(rows - 12, rows)])
    compare(layer, xd, rx, p, k, dtype, rows=sel)
    y = layer.forward(xd)
    # the split tiles' counters are back at zero, here and in the scratch array
    assert torch.equal(layer.forward(xd), y)
    for _ in range(2):
        z = torch.full_like(y, float("nan"))
        rc, msg = _noalloc(layer, xd, z)
        assert rc == 0, msg
        torch.cuda.synchronize()
        assert torch.equal(z, y)
    return layer, xd, y


@pytest.mark.parametrize("dtype,rows,D,H,up,down", ONE_EXPERT)
def test_one_expert(dtype, rows, D, H, up, down):
    layer, xd, y = check(rows, D, 1, 1, H, dtype, 800 + H)
    if not layer.uses_mfma:  # padded: the bits of gemm_rows' calls
        for n in (50, 1000):
            assert torch.equal(layer.forward(xd[:n]), y[:n]), n


@pytest.mark.parametrize("dtype,rows,D,E,k,H", EXPERTS)
def test_several_experts(dtype, rows, D, E, k, H):
    check(rows, D, E, k, H, dtype, 900 + H)
