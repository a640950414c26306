"""GEMMs of few rows and of widths that no tile divides (csrc/gemm_rows.hip,
the zero padding of csrc/gemm_mfma.hip and csrc/dispatch.hip).

Bars: compare() of tests/_gpu.py, against the f64 oracle and the oracle with
the kernels' storage roundings.
"""
import numpy as np
import pytest
import torch

from _common import rounded, small_case
from _gpu import compare, layer_from_tensors, to_device
import nomas_moe as nm
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


def run_case(rows, D, E, k, H, dtype, seed, s=0.0):
    print(f"rows={rows} D={D} E={E} k={k} H={H} {dtype} dense={s}", flush=True)
    t, x = small_case(rows, D, E, k, H, seed, dense=s > 0, router_std=0.5)
    layer = layer_from_tensors(t, dtype, D, H, E, k, s)
    rt, rx = rounded(t, x, dtype)
    p, dn = nm.workloads.oracle_params(rt, E)
    compare(layer, to_device(x, dtype), rx, p, k, dtype, shared_dense=s, dense=dn)
    return t, x, layer


# one expert takes every row: 16-, 32- and 64-row tiles full, one row short and one over
@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32, 33, 63, 65, 130])
def test_tile_edges(rows, dtype):
    run_case(rows, 256, 1, 1, 384, dtype, 500 + rows)


# D and H at the edges of K turns (128 or 64 columns), of 256-row weight tiles and of 16-byte chunks
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("D,H", [(8, 1), (64, 127), (72, 129), (248, 33), (264, 257), (520, 640), (256, 100)])
@pytest.mark.parametrize("rows", [5, 400])
def test_padded_widths(rows, D, H, dtype):
    run_case(rows, D, 3, 2, H, dtype, 600 + D + H, 0.5 if D == 72 else 0.0)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_padded_rows_do_not_depend_on_the_call(dtype):
    """Every row of a padded-width layer is the same bits in a call of 9,000 rows and of 3."""
    t, x = small_case(9000, 264, 2, 1, 700, 77)
    layer = layer_from_tensors(t, dtype, 264, 700, 2, 1)
    xd = to_device(x, dtype)
    y = layer.forward(xd)
    for rows in (3, 40, 200, 1500):
        assert torch.equal(layer.forward(xd[:rows]), y[:rows]), rows


def test_padded_non_finite_rows_stay_apart():
    """An infinite and a NaN input row leave the other rows' bits alone, and a
    layer of one hidden unit does not turn an infinity into NaN by its padding."""
    D, H, rows = 72, 1, 50
    ones = {f"ffn.{n}.weight": np.full(sh, 0.1, np.float32)
            for n, sh in (("gate", (H, D)), ("up", (H, D)), ("down", (D, H)))}
    layer = nm.FeedForward.from_source(nm.Weights.tensors_(ones, "f32"), "ffn", D, H)
    xd = torch.randn(rows, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    y = layer.forward(xd)
    bad = xd.clone()
    bad[3, 5] = float("inf")
    bad[40, 0] = float("nan")
    yb = layer.forward(bad)
    keep = [i for i in range(50) if i not in (3, 40)]
    assert torch.equal(yb[keep], y[keep])
    assert torch.isposinf(yb[3]).all() and torch.isnan(yb[40]).all()


def test_noalloc_in_pieces():
    """A no-allocation call whose padded buffers exceed the scratch array runs
    in row pieces: the same bits and routing as the allocating forward."""
    rows, D, E, k, H = 1_200_000, 8, 3, 1, 4
    t, _ = small_case(8, D, E, k, H, 79, router_std=0.5)
    layer = layer_from_tensors(t, "bf16", D, H, E, k)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(rows, D, device="cuda", generator=g).to(torch.bfloat16)
    y_ref = layer.forward(x)
    ref = layer.routing(rows)
    y = torch.full_like(y_ref, float("nan"))
    rc, msg = _noalloc(layer, x, y)
    assert rc == 0, msg
    torch.cuda.synchronize()
    assert torch.equal(y, y_ref)
    for a, b in zip(layer.routing(rows), ref):
        assert np.array_equal(a, b)
