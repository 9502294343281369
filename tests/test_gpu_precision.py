"""Cases where the size of one value must not cost another its bits (inputs that cancel, rows and channels of
very different size, gradients of small rows beside large ones) or the batch a row its bits (few rows against
the tiles); scratch, shapes and alignment that a path must take or refuse as every other path does."""

import numpy as np
import pytest
import torch

from _gpu_helpers import bf16_round, say
from oracle import dense, moe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [400, 401])
def test_int8_layer_multiplies_the_given_bf16_inputs(N):
    """Two input channels that cancel but for a component 2^-11 to 2^-14 of the rest: the int8 layer's products
    take x as given, so what is left comes out within the output's own rounding (h and y in bf16: 2^-8)."""
    import yggdrasil_amd

    d, F, E = 34, 48, 2
    g = np.random.default_rng(N)
    x = np.zeros((N, d, 8), np.float32)
    x[:, 0, 0] = x[:, 1, 0] = 256.0
    x[:, 0, 3] = g.uniform(0.02, 0.12, N)
    x = bf16_round(x)
    wu = np.zeros((E, F, d, 8), np.float32)
    wu[:, :, 0, 0] = g.uniform(0.5, 2.0, (E, F))
    wu[:, :, 1, 0] = -wu[:, :, 0, 0]
    wd = (g.standard_normal((E, d, F, 8)) / np.sqrt(8 * F)).astype(np.float32)
    zeros = np.zeros((E, F, 8), np.float32), np.zeros((E, d, 8), np.float32)
    lg = g.standard_normal((N, E)).astype(np.float32)
    cfg = yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=F, n_experts=E, top_k=1, activation="relu", dtype=torch.bfloat16,
                                     weight_format="int8", router="logits")
    layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
    layer.load_reference_weights(w_up=wu, b_up=zeros[0], w_down=wd, b_down=zeros[1])
    say(f"int8 layer, cancelling inputs, N={N}")
    out = layer.moe_forward(torch.from_numpy(x).cuda().bfloat16()[None], logits=torch.from_numpy(lg).cuda())[0]
    idx = layer.last_routing["topk_idx"].cpu().numpy()
    w = layer.last_routing["topk_w"].cpu().numpy()
    ref = dense.moe_layer(x, idx, w, moe.dequantize_int8(*moe.quantize_int8(wu)), zeros[0],
                          moe.dequantize_int8(*moe.quantize_int8(wd)), zeros[1], "relu")
    err = out.float().cpu().numpy() - ref
    assert np.linalg.norm(err) < 2.0 ** -7 * np.linalg.norm(ref)


def _bf16_layer(d, F, E, k, act="gelu", router="logits"):
    import yggdrasil_amd

    torch.manual_seed(d + F + E)
    cfg = yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=F, n_experts=E, top_k=k, activation=act, dtype=torch.bfloat16,
                                     weight_format="pauli", router=router)
    layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
    with torch.no_grad():
        for p in (layer.b_up, layer.b_down):
            p.normal_(0.0, 0.1)
    return layer


@pytest.mark.parametrize("N,d,F,E,k,act", [
    (1, 2, 2, 1, 1, "gelu"), (9, 16, 18, 3, 2, "relu"), (40, 18, 16, 4, 3, "sigmoid"), (17, 24, 40, 64, 2, "gelu"),
    (33, 66, 258, 2, 1, "gelu"), (16, 256, 1024, 64, 2, "gelu"), (64, 128, 512, 8, 2, "relu"), (160, 100, 302, 12, 4, "sigmoid"),
    (701, 34, 98, 5, 2, "gelu"), (300, 200, 798, 4, 2, "relu"), (1201, 10, 16, 3, 1, "gelu")])
def test_few_rows_equal_the_tiles(N, d, F, E, k, act):
    """bf16 Pauli layers: a call of few rows gives, bit for bit, what the separate products give (which take
    the 64 x 64 tiles at every size), on both sides of d_in = 16, where the tiles change."""
    from yggdrasil_amd import ops

    layer = _bf16_layer(d, F, E, k, act)
    x = torch.randn(1, N, d, 8, device="cuda").bfloat16()
    lg = torch.randn(N, E, device="cuda")
    lg[:, 0] -= 20.0 * (E > k)  # an expert without rows
    say(f"few rows against tiles N={N} d={d} F={F} E={E} k={k} {act}")
    out = layer.moe_forward(x, logits=lg)
    prep = layer._get_prepared()
    r = ops.route(lg, k)
    h = ops.pauli_grouped_linear(ops.pauli_rows_from_blade(x[0]), prep["w_up"], r.offsets, prep["b_up"], act,
                                 gather=r.perm, x_layout="pauli", y_layout="pauli")
    y = ops.pauli_grouped_linear(h, prep["w_down"], r.offsets, prep["b_down"], "none", x_layout="pauli",
                                 y_layout="blade", out_dtype=torch.bfloat16)
    assert torch.equal(out[0], ops.combine(y, r))


@pytest.mark.parametrize("d,F,E,k", [(128, 512, 32, 2), (64, 130, 3, 1), (16, 32, 4, 2)])
def test_bf16_rows_do_not_depend_on_the_batch(d, F, E, k):
    """A token's output row is the same bits in a batch of 1, 7, 500, 900 and 3000 tokens."""
    layer = _bf16_layer(d, F, E, k)
    x = torch.randn(1, 3000, d, 8, device="cuda").bfloat16()
    lg = torch.randn(3000, E, device="cuda")
    say(f"batch invariance d={d} F={F} E={E} k={k}")
    full = layer.moe_forward(x, logits=lg)
    for n in (1, 7, 500, 900):
        assert torch.equal(layer.moe_forward(x[:, :n].contiguous(), logits=lg[:n].contiguous()), full[:, :n])


@pytest.mark.parametrize("N,d,E,k", [(64, 256, 8, 2), (256, 64, 8, 2), (1024, 40, 64, 4)])
def test_route_energy_needs_no_scratch_up_to_1024_tokens(N, d, E, k):
    """The C entry up to 1024 tokens: no workspace, a scratch that it does not touch, the outputs of the
    same call in two steps."""
    from yggdrasil_amd import ops
    from yggdrasil_amd._native import check, lib, ptr, stream_handle

    torch.manual_seed(N)
    x = torch.randn(N, d, 8, device="cuda")
    rw, rb = torch.randn(E, 4, device="cuda"), torch.randn(E, device="cuda")
    out = {n: torch.empty(s, device="cuda", dtype=t) for n, s, t in (
        ("idx", (N, k), torch.int32), ("w", (N, k), torch.float32), ("counts", (E,), torch.int32),
        ("offsets", (E + 1,), torch.int32), ("perm", (N * k,), torch.int32), ("slot", (N, k), torch.int32))}
    scratch = torch.full((N * E,), -7.0, device="cuda")
    say(f"route_energy without workspace N={N} d={d} E={E}")
    check(lib().ygg_route_energy(ptr(x), 0, N, d, ptr(rw), ptr(rb), E, k, ptr(out["idx"]), ptr(out["w"]),
                                 ptr(out["counts"]), ptr(out["offsets"]), ptr(out["perm"]), ptr(out["slot"]),
                                 ptr(scratch), None, 0, stream_handle(x.device)), "route_energy")
    assert (scratch == -7.0).all()
    ref = ops.route(ops.router_energy_logits(x, rw, rb), k)
    same = (out["idx"] == ref.topk_idx).all(dim=1)  # (the two sum in another order: ties may differ)
    assert same.float().mean().item() > 0.98
    assert (out["w"] - ref.topk_w)[same].abs().max().item() < 1e-5
    assert int(out["counts"].sum()) == N * k and torch.equal(out["offsets"][1:], out["counts"].cumsum(0).int())
    tok = torch.arange(N, device="cuda").repeat_interleave(k)
    assert torch.equal(out["perm"][out["slot"].flatten().long()].long(), tok)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,d,E,k", [(70, 256, 8, 2), (203, 66, 8, 3), (256, 64, 64, 2), (1024, 40, 33, 4)])
def test_energy_logits_of_the_layer_and_the_entry_are_the_same(N, d, E, k, dtype):
    """From these sizes on a layer takes the grade-energy logits in a launch of its own, the entry never does:
    the same sums in the same order, so the same weights bit for bit, every token."""
    import yggdrasil_amd
    from yggdrasil_amd import ops

    cfg = yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=16, n_experts=E, top_k=k, dtype=dtype, router="energy")
    layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
    with torch.no_grad():
        layer.router_weight.normal_()
        layer.router_bias.normal_()
    x = torch.randn(1, N, d, 8, device="cuda").to(dtype)
    say(f"energy logits N={N} d={d} E={E} {dtype}")
    with torch.no_grad():
        layer.moe_forward(x)
    r = ops.route_energy(x[0], layer.router_weight.detach(), layer.router_bias.detach(), k)
    got = layer.last_routing
    assert torch.equal(got["topk_idx"], r.topk_idx) and torch.equal(got["topk_w"], r.topk_w)
    assert torch.equal(got["counts"], r.counts) and torch.equal(got["offsets"], r.offsets)


def _split(*sizes):
    """The case runs on the units it means to test."""
    from yggdrasil_amd._native import lib

    assert (lib().ygg_f32_product_split if len(sizes) == 3 else lib().ygg_f32_layer_split)(*sizes) == 1


def _rows_rel(got, ref):
    """The largest relative 2-norm error of a row."""
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    got, ref = got.reshape(got.shape[0], -1), ref.reshape(ref.shape[0], -1)
    return float((np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)).max())


# 24 bits of each operand, sums of up to 1000 fp32 terms of random sign: 2^-24 sqrt(1000) of a row's norm at most
FP32_ROW = 2e-6


@pytest.mark.parametrize("M,K,N", [(64, 128, 6400), (70, 130, 6000), (129, 33, 3300)])
def test_geom_matmul_keeps_small_inputs_beside_large_ones(M, K, N):
    """Output rows whose weights are zero on the large inputs depend on the small ones, 2^-28 below, alone."""
    from yggdrasil_amd import ops

    _split(N, K, M)
    g = np.random.default_rng(M)
    a = g.standard_normal((M, K, 8)).astype(np.float32)
    b = g.standard_normal((K, N, 8)).astype(np.float32)
    a[::2, :K // 2] = 0.0
    b[:K // 2] *= np.float32(2.0 ** 28)
    say(f"geom_matmul, small inputs beside large ones M={M} K={K} N={N}")
    out = ops.geom_matmul(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()).cpu().numpy()
    ref = np.transpose(dense.linear(np.transpose(b, (1, 0, 2)), a), (1, 0, 2))
    assert _rows_rel(out, ref) < FP32_ROW


def _lopsided(N, d, F, E, scale):
    """An expert's first token is `scale` times the others and lies in the first half of the inputs, from which the
    second half of the hidden channels has no weights."""
    g = np.random.default_rng(N + F)
    x = g.standard_normal((N, d, 8)).astype(np.float32)
    lg = g.standard_normal((N, E)).astype(np.float32)
    big = [int(np.flatnonzero(lg.argmax(1) == e)[0]) for e in range(E)]
    x[big] *= np.float32(scale)
    x[big, d // 2:] = 0.0
    wu = (g.standard_normal((E, F, d, 8)) / np.sqrt(8 * d)).astype(np.float32)
    wu[:, F // 2:, :d // 2] = 0.0
    wd = (g.standard_normal((E, d, F, 8)) / np.sqrt(8 * F)).astype(np.float32)
    return g, x, lg, big, wu, wd, np.zeros((E, F, 8), np.float32), np.zeros((E, d, 8), np.float32)


@pytest.mark.parametrize("N,F", [(4096, 128), (20000, 250)])
def test_layer_and_gradients_keep_small_rows_beside_large_ones(N, F):
    """A token 2^25 times the others, in x and in the output's gradient: weight gradients to which it adds exact
    zeros keep the other tokens' to fp32, and the other tokens' outputs and gradients theirs.  (The weight gradients
    take the fp32 units in the smaller case, the bf16 ones in the larger.)"""
    import yggdrasil_amd

    d, E = 128, 2
    _split(N, d, F, E, 1)
    g, x, lg, big, wu, wd, bu, bd = _lopsided(N, d, F, E, 2.0 ** 25)
    dout = g.standard_normal((N, d, 8)).astype(np.float32)
    dout[big] *= np.float32(2.0 ** 25)
    cfg = yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=F, n_experts=E, top_k=1, activation="gelu", router="logits")
    layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
    layer.load_reference_weights(w_up=wu, b_up=bu, w_down=wd, b_down=bd)
    say("fp32 layer, one token 2^25 times the others")
    xt = torch.from_numpy(x).cuda()[None].requires_grad_(True)
    out = layer.moe_forward(xt, logits=torch.from_numpy(lg).cuda())
    grads = torch.autograd.grad(out, (xt, layer.w_up, layer.w_down), torch.from_numpy(dout).cuda()[None])
    dx, dwu, dwd = (t.cpu().numpy() for t in grads)
    idx = layer.last_routing["topk_idx"].cpu().numpy()
    w = layer.last_routing["topk_w"].cpu().numpy()
    ref = dense.moe_layer(x, idx, w, wu, bu, wd, bd, "gelu")
    rdx, rwu, _, rwd, _ = dense.moe_layer_backward(x, idx, w, wu, bu, wd, bd, dout, "gelu")
    # two products in turn and the activation's fast exponential (2^-21 of a component)
    assert _rows_rel(out[0].detach().cpu().numpy(), ref) < 2 * FP32_ROW
    assert _rows_rel(dx[0], rdx) < 2 * FP32_ROW
    for e in range(E):
        # sums over 10000 tokens of terms of random sign, 384 at a time: below 2^-24 sqrt(1000) of a row's norm, and
        # the products' errors
        assert _rows_rel(dwd[e][:, F // 2:], rwd[e][:, F // 2:]) < 2 * FP32_ROW  # (the large token's h is zero there)
        assert _rows_rel(dwu[e][:, d // 2:], rwu[e][:, d // 2:]) < 2 * FP32_ROW  # (and its x there)
        assert _rows_rel(dwd[e][:, :F // 2], rwd[e][:, :F // 2]) < 2 * FP32_ROW


@pytest.mark.parametrize("k", [1, 2])
def test_layer_with_non_finite_rows(k):
    """Tokens with a NaN or an infinity: their rows are not finite, every other row is as without them."""
    import yggdrasil_amd

    N, d, F, E = 3000, 129, 130, 3
    _split(N, d, F, E, k)
    torch.manual_seed(k)
    layer = yggdrasil_amd.CliffordMoELayer(
        yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=F, n_experts=E, top_k=k, router="logits"), device="cuda")
    x, lg = torch.randn(1, N, d, 8, device="cuda"), torch.randn(N, E, device="cuda")
    x[0, 11] = 0.0
    bad = x.clone()
    bad[0, 7, 3, 2] = float("nan")
    bad[0, 2222, 99, 0] = float("inf")
    say(f"fp32 layer, non-finite tokens, k={k}")
    with torch.no_grad():
        out, out_bad = layer.moe_forward(x, logits=lg), layer.moe_forward(bad, logits=lg)
    keep = torch.ones(N, dtype=torch.bool, device="cuda")
    keep[[7, 2222]] = False
    assert torch.isfinite(out).all() and torch.equal(out[0][keep], out_bad[0][keep])
    assert not torch.isfinite(out_bad[0, [7, 2222]]).flatten(1).all(dim=1).any()
    # a NaN in one token's gradient reaches the weights of its experts only
    xt = x.clone().requires_grad_(True)
    go = torch.randn_like(x)
    params = (layer.w_up, layer.b_up, layer.w_down, layer.b_down)
    ref = torch.autograd.grad(layer.moe_forward(xt, logits=lg), params, go)
    go[0, 7, 5, 1] = float("nan")
    got = torch.autograd.grad(layer.moe_forward(xt, logits=lg), params, go)
    hit = set(layer.last_routing["topk_idx"][7].tolist())
    for a, b in zip(ref, got):
        for e in range(E):
            assert torch.isfinite(b[e]).all() == (e not in hit)
            assert e in hit or torch.equal(a[e], b[e])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name,shape", [("router_weight", (3, 4)), ("router_weight", (4, 3)), ("router_bias", (3,)),
                                        ("w_up", (4, 8, 10, 8)), ("w_down", (4, 16, 16, 8)), ("b_up", (3, 16, 8)),
                                        ("b_down", (4, 14, 8))])
def test_replaced_parameters_of_another_shape_are_refused(name, shape, dtype):
    """A parameter replaced by one of another shape raises before its pointer reaches a kernel."""
    import yggdrasil_amd

    layer = yggdrasil_amd.CliffordMoELayer(
        yggdrasil_amd.MoEHLMConfig(d_model=10, d_ff=16, n_experts=4, top_k=2, dtype=dtype), device="cuda")
    setattr(layer, name, torch.nn.Parameter(torch.zeros(shape, device="cuda")))
    say(f"{name} {shape}")
    with torch.no_grad(), pytest.raises(ValueError, match=name):
        layer.moe_forward(torch.randn(1, 5, 10, 8, device="cuda").to(dtype))


def test_weight_preparation_of_any_aligned_floats():
    """Weights that are a view into a flat buffer, four bytes off: both layouts as of an aligned copy."""
    from yggdrasil_amd import ops

    flat = torch.randn(3 * 37 * 50 * 8 + 1, device="cuda")
    w = flat[1:].view(3, 37, 50, 8)
    assert w.data_ptr() % 16 == 4
    say("weights four bytes off")
    assert torch.equal(ops.prepare_weights(w, "pauli_f32").data, ops.prepare_weights(w.clone(), "pauli_f32").data)
    assert torch.equal(ops.prepare_adjoint_weights(w).data, ops.prepare_adjoint_weights(w.clone()).data)
