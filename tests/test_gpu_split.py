"""fp32 products on the bf16 MFMA units (operands as three bf16 parts) against float64.

The parts hold the 24 bits of a value.  Error model of an output element: the products of parts that are
left out are at most 2^-23 of a product, and the sums are fp32, one rounding of a full sum per eight inputs
and those of the small sums, 2^-24 of partial sums of random terms.  In the 2-norm that stays below
(2^-23 + 2^-24 sqrt(d_in / 8)) of the result: 3.6e-7 for d_in = 128, 6e-7 for 512; the bound used is 2e-6, which
the fp32 MFMA units' sums (4 d_in terms in a chain of pairs) meet too.
"""

import numpy as np
import pytest
import torch

from _gpu_helpers import say
from oracle import dense

pytestmark = pytest.mark.gpu

TOL = 2e-6


def _rel(got, ref):
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    return float(np.linalg.norm(got - ref) / np.linalg.norm(ref))


def _gm(a, b):
    from yggdrasil_amd import ops

    return ops.geom_matmul(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()).cpu().numpy()


def _truth(a, b):
    return np.transpose(dense.linear(np.transpose(b, (1, 0, 2)), a), (1, 0, 2))


def _split_product(rows, d_in, d_out):
    from yggdrasil_amd._native import lib

    return lib().ygg_f32_product_split(rows, d_in, d_out) == 1


@pytest.mark.parametrize("M,K,N", [(64, 128, 6400), (65, 129, 6333), (130, 136, 3300), (513, 143, 800), (66, 255, 6300),
                                   (100, 32, 4100), (13, 33, 31600), (8191, 41, 51)])
def test_geom_matmul_sizes(M, K, N):
    """Sizes from which the split product runs, on and off its tiles (64 x 64, blocks of 8 inputs)."""
    assert _split_product(N, K, M)
    g = np.random.default_rng(M + K + N)
    a = (g.standard_normal((M, K, 8)) / np.sqrt(8 * K)).astype(np.float32)
    b = g.standard_normal((K, N, 8)).astype(np.float32)
    say(f"split geom_matmul M={M} K={K} N={N}")
    assert _rel(_gm(a, b), _truth(a, b)) < TOL


def test_geom_matmul_scales_and_non_finite():
    """Rows and channels over 200 binades, zero rows, entries 2^-20 below their row's largest, and rows
    with an infinity or NaN: those give non-finite rows, and every other row is as without them."""
    g = np.random.default_rng(4)
    M, K, N = 70, 130, 6000
    assert _split_product(N, K, M)
    a = (g.standard_normal((M, K, 8)) / np.sqrt(8 * K)).astype(np.float32)
    b = g.standard_normal((K, N, 8)).astype(np.float32)
    a *= np.ldexp(1.0, g.integers(-60, 40, (M, 1, 1))).astype(np.float32)
    b *= np.ldexp(1.0, g.integers(-60, 40, (1, N, 1))).astype(np.float32)
    b[:40] *= np.float32(2.0 ** -20)
    b[:, 17] = 0.0
    bad = b.copy()
    bad[3, 100, 2] = np.inf
    bad[5, 2000, 0] = np.nan
    say("split geom_matmul scales, non-finite")
    ref = _truth(a, b)
    out, out_bad = _gm(a, b), _gm(a, bad)
    # sqrt(8 K) random terms of the largest size in the row and the channel
    scale = np.abs(a).max(axis=(1, 2))[:, None] * np.abs(b).max(axis=(0, 2))[None, :] * np.sqrt(8 * K)
    err = np.linalg.norm(out - ref, axis=2)
    assert np.isfinite(out).all() and not out[:, 17].any()
    assert (err <= 1e-6 * scale).all()
    assert not np.isfinite(out_bad[:, [100, 2000]]).any()
    keep = np.ones(N, bool)
    keep[[100, 2000]] = False
    assert np.array_equal(out_bad[:, keep], out[:, keep])


@pytest.mark.parametrize("N,d,F,E,k,act,empty", [(1700, 128, 256, 5, 2, "gelu", False), (3300, 133, 141, 3, 1, "sigmoid", True),
                                                 (1300, 150, 128, 8, 4, "relu", False)])
def test_layer(N, d, F, E, k, act, empty):
    """The fp32 layer with both products split: widths off the blocks of 8, an expert without rows, odd row
    counts, tokens over many binades, biases and a residual."""
    import yggdrasil_amd

    g = np.random.default_rng(N + d)
    x = g.standard_normal((N, d, 8)).astype(np.float32) * np.ldexp(1.0, g.integers(-12, 4, (N, 1, 1))).astype(np.float32)
    lg = g.standard_normal((N, E)).astype(np.float32)
    if empty:
        lg[:, 1] = -30.0
    wu = (g.standard_normal((E, F, d, 8)) / np.sqrt(8 * d)).astype(np.float32)
    wd = (g.standard_normal((E, d, F, 8)) / np.sqrt(8 * F)).astype(np.float32)
    bu, bd = ((0.1 * g.standard_normal(s)).astype(np.float32) for s in ((E, F, 8), (E, d, 8)))
    res = g.standard_normal((N, d, 8)).astype(np.float32)
    cfg = yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=F, n_experts=E, top_k=k, activation=act, router="logits")
    layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
    layer.load_reference_weights(w_up=wu, b_up=bu, w_down=wd, b_down=bd)
    say(f"split layer N={N} d={d} F={F} E={E} k={k} {act}")
    with torch.no_grad():
        out = layer.moe_forward(torch.from_numpy(x).cuda()[None], logits=torch.from_numpy(lg).cuda(),
                                residual=torch.from_numpy(res).cuda()[None])[0].cpu().numpy()
    idx = layer.last_routing["topk_idx"].cpu().numpy()
    w = layer.last_routing["topk_w"].cpu().numpy()
    ref = dense.moe_layer(x, idx, w, wu, bu, wd, bd, act, residual=res)
    # two products in turn (their errors add), the activation's fast exponential (2^-21)
    assert _rel(out, ref) < 2 * TOL
    assert _rel(out - res, ref - res) < 4 * TOL  # (and the residual's rounding, 2^-24 of a larger sum)


@pytest.mark.parametrize("rows,d_in,d_out,bias,dtype", [
    (6400, 128, 64, True, "f32"), (1637, 131, 257, False, "f32"), (6399, 127, 65, True, "f32"),  # split product
    (6399, 128, 64, True, "f32"), (1, 1, 1, True, "f32"), (33, 300, 5, False, "f32"),  # fp32 MFMA product
    (200, 9, 40, True, "bf16"), (17, 128, 33, False, "bf16"), (0, 16, 8, True, "f32")])
def test_clifford_linear_module(rows, d_in, d_out, bias, dtype):
    """The module on each of its paths, from a strided and from a misaligned input."""
    import yggdrasil_amd

    g = np.random.default_rng(rows + d_in)
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    x = torch.from_numpy(g.standard_normal((rows, d_in, 8)).astype(np.float32)).to(dt)
    w = (g.standard_normal((d_out, d_in, 8)) / np.sqrt(8 * d_in)).astype(np.float32)
    b = g.standard_normal((d_out, 8)).astype(np.float32)
    lin = yggdrasil_amd.CliffordLinear(d_in, d_out, bias=bias, dtype=dt, device="cuda")
    with torch.no_grad():
        lin.weight.copy_(torch.from_numpy(w))
        if bias:
            lin.bias.copy_(torch.from_numpy(b))
    say(f"CliffordLinear {rows} x {d_in} -> {d_out} {dtype}")
    assert _split_product(rows, d_in, d_out) == (rows * d_out >= 100 * 64 * 64 and d_in >= 32)
    shifted = torch.empty(rows * d_in * 8 + 1, dtype=dt, device="cuda")[1:].view(rows, d_in, 8)
    strided = torch.empty((rows, 2 * d_in, 8), dtype=dt, device="cuda")[:, ::2]
    shifted.copy_(x)
    strided.copy_(x)
    y = lin(x.cuda())
    assert y.shape == (rows, d_out, 8) and y.dtype == dt
    assert torch.equal(lin(shifted), y) and torch.equal(lin(strided), y)
    assert torch.equal(lin(x.cuda()[None])[0], y)
    if rows:
        w_held = torch.from_numpy(w).to(dt).double().numpy()
        ref = dense.linear(x.double().numpy(), w_held, b if bias else None)
        # bf16: the output's rounding, 2^-9 of each element at most
        assert _rel(y.double().cpu().numpy(), ref) < (TOL if dtype == "f32" else 2.0 ** -9)


@pytest.mark.parametrize("N,d,F,E,k,act,router", [(3300, 133, 150, 3, 1, "gelu", "logits"),
                                                  (1700, 128, 260, 5, 2, "sigmoid", "energy"),
                                                  (1301, 150, 128, 8, 4, "relu", "logits"),
                                                  (1201, 261, 180, 2, 2, "gelu", "logits")])
def test_layer_backward(N, d, F, E, k, act, router):
    """Gradients through the split products and weight gradients: widths off every block, an expert without
    rows, chunks with odd tails, tokens over many binades (rows of one weight-gradient sum have different
    scales), one token of zeros."""
    import yggdrasil_amd

    g = np.random.default_rng(N + d)
    x = g.standard_normal((N, d, 8)).astype(np.float32) * np.ldexp(1.0, g.integers(-9, 4, (N, 1, 1))).astype(np.float32)
    x[7] = 0.0
    lg = g.standard_normal((N, E)).astype(np.float32)
    if E == 3:
        lg[:, 1] = -30.0
    wu = (g.standard_normal((E, F, d, 8)) / np.sqrt(8 * d)).astype(np.float32)
    wd = (g.standard_normal((E, d, F, 8)) / np.sqrt(8 * F)).astype(np.float32)
    bu, bd = ((0.1 * g.standard_normal(s)).astype(np.float32) for s in ((E, F, 8), (E, d, 8)))
    dout = g.standard_normal((N, d, 8)).astype(np.float32) * np.ldexp(1.0, g.integers(-9, 4, (N, 1, 1))).astype(np.float32)
    cfg = yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=F, n_experts=E, top_k=k, activation=act, router=router)
    layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
    layer.load_reference_weights(w_up=wu, b_up=bu, w_down=wd, b_down=bd)
    say(f"split backward N={N} d={d} F={F} E={E} k={k} {act}")
    xt = torch.from_numpy(x).cuda()[None].requires_grad_(True)
    out = layer.moe_forward(xt, logits=torch.from_numpy(lg).cuda() if router == "logits" else None)
    grads = torch.autograd.grad(out, (xt, layer.w_up, layer.b_up, layer.w_down, layer.b_down),
                                torch.from_numpy(dout).cuda()[None])
    idx = layer.last_routing["topk_idx"].cpu().numpy()
    w = layer.last_routing["topk_w"].cpu().numpy()
    assert _rel(out[0].detach().cpu().numpy(), dense.moe_layer(x, idx, w, wu, bu, wd, bd, act)) < 2 * TOL
    ref = dense.moe_layer_backward(x, idx, w, wu, bu, wd, bd, dout, act)
    for name, got, want in zip(("dx", "dw_up", "db_up", "dw_down", "db_down"), grads, ref):
        got = got.cpu().numpy().reshape(want.shape)
        # the sums' error of two products and the activation's derivative in fp32
        assert np.isfinite(got).all() and _rel(got, want) < 4 * TOL, (name, _rel(got, want))
        if E == 3 and name != "dx":
            assert not got[1].any()
