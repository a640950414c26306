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
from gemm_cases import DENSE
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


# widths at the edges of the 32-wide steps that gemm_rows walks and of the 32 hidden
# units of its gate/up tiles: it skips all other padding
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("D,H", [(24, 31), (32, 32), (40, 33), (96, 64), (136, 65), (160, 224)])
@pytest.mark.parametrize("rows", [3, 700])
def test_padding_that_is_skipped(rows, D, H, dtype):
    run_case(rows, D, 3, 2, H, dtype, 650 + D + H, 0.5 if D == 40 else 0.0)


# gate/up on 256-row tiles and down on 64-row ones (two tile tables)
@pytest.mark.parametrize("D,H,dtype", [(1024, 2688, "bf16"), (1000, 2667, "bf16"), (512, 2048, "f32")])
def test_gemms_of_different_tile_heights(D, H, dtype):
    run_case(1111, D, 6, 2, H, dtype, 700 + D)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
def test_padded_rows_do_not_depend_on_the_call(dtype):
    """Every row of a padded-width layer is the same bits in a call of 9,000 rows (gate/up on
    256-row tiles) and of 3."""
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


# rows, D, H: gemm_rows' tiles (32 and 64 rows; padded) and gemm_mfma's (whole, gate/up or
# down split along K, padded)
@pytest.mark.parametrize("rows,D,H", [(70, 256, 128), (3000, 512, 256), (3000, 200, 72)] +
                         [c[1:4] for c in DENSE])
def test_f32_values_that_have_no_finite_planes(rows, D, H):
    """f32 rows with an infinity, a NaN or a value that rounds past bf16's
    largest, and weights of that size: each row as f32 arithmetic has it, the
    other rows' bits unchanged.  The bar on the finite values is that of f32
    sums of one large term and D small ones (a few ulps)."""
    big = np.float32(3.4e38)

    def ffn(gate):
        w = {"ffn.gate.weight": gate, "ffn.up.weight": np.full((H, D), 1e-20, np.float32),
             "ffn.down.weight": np.full((D, H), 1e-3, np.float32)}
        return nm.FeedForward.from_source(nm.Weights.tensors_(w, "f32"), "ffn", D, H)

    layer = ffn(np.full((H, D), 1e-20, np.float32))
    x = torch.randn(rows, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    y = layer.forward(x)
    bad = x.clone()
    bad[3, 5] = float("inf")
    bad[40, 0] = float("nan")
    bad[60] = 0.0
    bad[60, 7] = float(big)
    yb = layer.forward(bad)
    keep = [i for i in range(rows) if i not in (3, 40, 60)]
    assert torch.equal(yb[keep], y[keep])
    assert torch.isposinf(yb[3]).all() and torch.isnan(yb[40]).all()
    want = (float(big) * float(np.float32(1e-20))) ** 2 * H * float(np.float32(1e-3))
    # (H equal terms: each of at most H adds rounds by 2^-24 of the sum)
    assert torch.allclose(yb[60].double(), torch.full((D,), want, device="cuda", dtype=torch.float64),
                          rtol=max(2e-6, H * 2.0 ** -24))
    # one weight of 3.4e38 in every hidden unit's gate, met by x = 1e-30
    gate = np.full((H, D), 1e-3, np.float32)
    gate[:, 2] = big
    x[:, 2] = 1e-30
    got = ffn(gate).forward(x).double()
    g = x.double() @ torch.from_numpy(gate).cuda().double().T
    u = x.double().sum(1, keepdim=True) * float(np.float32(1e-20))
    want = (g * torch.sigmoid(g) * u).sum(1, keepdim=True) * float(np.float32(1e-3))
    assert torch.isfinite(got).all()
    assert (got - want).norm() <= 1e-5 * want.norm() * np.sqrt(D)  # want: (rows, 1), got: its D columns


def test_f32_repaired_rows_do_not_depend_on_the_call():
    """A gate weight and a down weight of 3.4e38 make one hidden unit and one
    output column of every row sums that the planes cannot hold.  Those values
    are made again, every other one keeps its bits: a row is the same in a call
    of 9,000 rows (256-row tiles in both GEMMs) and in small ones."""
    rows, D, H = 9000, 1000, 2667
    g = torch.Generator(device="cuda").manual_seed(9)

    def randn(*shape, std):
        return (torch.randn(*shape, generator=g, device="cuda") * std).cpu().numpy()

    w = {"ffn.gate.weight": randn(H, D, std=D ** -0.5), "ffn.up.weight": randn(H, D, std=D ** -0.5),
         "ffn.down.weight": randn(D, H, std=H ** -0.5), "ffn.up.bias": randn(H, std=0.1)}
    w["ffn.gate.weight"][5, 2] = 3.4e38
    w["ffn.up.weight"][9] = 0.0
    w["ffn.up.bias"][9] = 1e-30
    w["ffn.down.weight"][7, 9] = 3.4e38
    zeros = {"ffn.gate.bias": np.zeros(H, np.float32), "ffn.down.bias": np.zeros(D, np.float32)}
    layer = nm.FeedForward.from_source(nm.Weights.tensors_({**w, **zeros}, "f32"), "ffn", D, H)
    x = torch.randn(rows, D, generator=g, device="cuda")
    x[:, 2] = 1e-30
    y = layer.forward(x)
    for n in (40, 700):
        assert torch.equal(layer.forward(x[:n]), y[:n]), n
    # and right: every column to f32 sums of about 3,000 terms
    t = {k: torch.from_numpy(v).cuda().double() for k, v in w.items()}
    xd = x[:200].double()
    gate, up = xd @ t["ffn.gate.weight"].T, xd @ t["ffn.up.weight"].T + t["ffn.up.bias"]
    want = (gate * torch.sigmoid(gate) * up) @ t["ffn.down.weight"].T
    err = (y[:200].double() - want).norm(dim=0) / want.norm(dim=0)
    print(f"  worst column {float(err.max()):.2e}", flush=True)
    assert err.max() <= 5e-6


# calls of few rows (whole tiles and padded), and of 256-row tiles
@pytest.mark.parametrize("rows,D,H", [(70, 256, 128), (70, 264, 100), (9000, 1024, 2048), (9000, 1000, 2667)])
@pytest.mark.parametrize("exp", [-112, -119, -126])
@pytest.mark.parametrize("tiny", ["x", "up", "down", "up, one large", "down, one large"])
def test_f32_tiny_values(tiny, exp, rows, D, H):
    """Activations or weights around 2^exp, down to subnormal ones: as exact as f32
    sums of values near 1 (TIGHT's 5e-6; at 2^-126 the results' own last
    place is up to 2^-22 of them, 2.4e-7).  One weight of 3e38 among them, on
    an input that is zero, changes nothing."""
    g = torch.Generator(device="cuda").manual_seed(10)

    def randn(*shape, std):
        return (torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64) * std).float().cpu().numpy()

    sc = 2.0 ** exp
    w = {"ffn.gate.weight": np.zeros((H, D), np.float32), "ffn.gate.bias": np.ones(H, np.float32),
         "ffn.up.weight": randn(H, D, std=D ** -0.5 * (sc if tiny[:2] == "up" else 1)),
         "ffn.up.bias": np.zeros(H, np.float32),
         "ffn.down.weight": randn(D, H, std=H ** -0.5 * (sc if tiny[:4] == "down" else 1)),
         "ffn.down.bias": np.zeros(D, np.float32)}
    x = torch.from_numpy(randn(rows, D, std=sc if tiny == "x" else 1)).cuda()
    if tiny == "up, one large":
        w["ffn.up.weight"][3, 4] = 3e38
        x[:, 4] = 0.0
    if tiny == "down, one large":
        w["ffn.up.weight"][6] = 0.0
        w["ffn.down.weight"][5, 6] = 3e38
    y = nm.FeedForward.from_source(nm.Weights.tensors_(w, "f32"), "ffn", D, H).forward(x)[:200].double()
    t = {k: torch.from_numpy(v).cuda().double() for k, v in w.items()}
    want = (x[:200].double() @ t["ffn.up.weight"].T * torch.sigmoid(torch.ones(1).double().cuda())) @ t["ffn.down.weight"].T
    err = float((y - want).norm() / want.norm())
    print(f"  {tiny} 2^{exp} {rows} x {D} x {H}: {err:.2e}", flush=True)
    assert err <= 5e-6


@pytest.mark.parametrize("shift", [0, 64, -64])
def test_host_output_over_the_input(shift):
    """A pinned host output that is the input, or overlaps it some rows on."""
    rows, D = 20_000, 264
    t, x = small_case(rows, D, 4, 1, 96, 82)
    layer = layer_from_tensors(t, "f32", D, 96, 4, 1)
    want = layer.forward(to_device(x, "f32")).cpu()
    buf = torch.empty(rows + 64, D, pin_memory=True)
    src = buf[64:] if shift < 0 else buf[:rows]
    dst = buf[:rows] if shift < 0 else buf[shift:shift + rows]
    src.copy_(torch.from_numpy(x))
    layer.forward(src, out=dst)
    assert torch.equal(dst, want)


def test_noalloc_in_pieces():
    """A no-allocation call whose padded buffers exceed the scratch array runs
    in row pieces: the same bits and routing as the allocating forward."""
    rows, D, E, k, H = 2_000_000, 8, 3, 1, 4
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


# more 64-row chunks than CUs, two dispatch blocks on a CU: rows of one 512-byte slab
# (padded, whole, and more x than the L2 caches hold) and of two
@pytest.mark.parametrize("rows,D,E,k,dtype", [(16448, 72, 6, 2, "f32"), (17000, 128, 40, 5, "bf16"), (16500, 128, 3, 1, "f32"),
                                              (70000, 256, 4, 1, "bf16"), (70001, 248, 4, 2, "bf16"), (17000, 288, 6, 2, "bf16")])
def test_dispatch_two_blocks_a_cu(rows, D, E, k, dtype):
    t, x = small_case(rows, D, E, k, 24, 690 + D, router_std=0.5)
    layer = layer_from_tensors(t, dtype, D, 24, E, k)
    rt, rx = rounded(t, x, dtype)
    p, dn = nm.workloads.oracle_params(rt, E)
    compare(layer, to_device(x, dtype), rx, p, k, dtype, rows=np.unique(np.r_[np.arange(0, rows, 61), rows - 1]))


def test_stage_times_of_a_call_in_pieces():
    """The stage times of a call in row pieces are those of the whole call: about a
    forward's in one piece (a mean over the pieces would be half of it or less)."""
    rows, D, E, k, H = 2_000_000, 8, 3, 1, 4
    t, _ = small_case(8, D, E, k, H, 84, router_std=0.5)
    layer = layer_from_tensors(t, "bf16", D, H, E, k)
    x = torch.randn(rows, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(8)).to(torch.bfloat16)
    y = torch.empty_like(x)
    host = x.cpu()

    def gemm_ms(call):
        call()
        layer.set_profiling(True)
        for _ in range(3):
            call()
        torch.cuda.synchronize()
        st = layer.stage_times()
        layer.set_profiling(False)
        return st["gemm_gate_up"] + st["gemm_down"] + st["router"]

    one = gemm_ms(lambda: layer.forward(x, out=y))
    for name, call in (("no allocation", lambda: _noalloc(layer, x, y)), ("host tensor", lambda: layer.forward(host))):
        ms = gemm_ms(call)
        print(f"  {name}: {ms:.3f} ms, in one piece {one:.3f} ms", flush=True)
        assert ms >= 0.75 * one, name


@pytest.mark.parametrize("shift", [0, 64, -64])
def test_noalloc_in_pieces_output_over_the_input(shift):
    """y is x, or overlaps it some rows on: every piece reads rows of x that
    no earlier piece has written."""
    rows, D, E, k, H = 2_000_000, 8, 3, 1, 4
    t, _ = small_case(8, D, E, k, H, 83, router_std=0.5)
    layer = layer_from_tensors(t, "bf16", D, H, E, k)
    g = torch.Generator(device="cuda").manual_seed(6)
    x = torch.randn(rows, D, device="cuda", generator=g).to(torch.bfloat16)
    want = layer.forward(x)
    ref = layer.routing(rows)
    buf = torch.empty(rows + 64, D, dtype=torch.bfloat16, device="cuda")
    src = buf[64:] if shift < 0 else buf[:rows]
    dst = buf[:rows] if shift < 0 else buf[shift:shift + rows]
    src.copy_(x)
    rc, msg = _noalloc(layer, src, dst)
    assert rc == 0, msg
    torch.cuda.synchronize()
    assert torch.equal(dst, want)
    for a, b in zip(layer.routing(rows), ref):
        assert np.array_equal(a, b)
