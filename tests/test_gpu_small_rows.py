"""bf16 Pauli layers of few rows (products that stream the weights), the routing's paths by batch size, weight
gradients of few rows and int8 layers of more than decode size."""

import numpy as np
import pytest
import torch

from _gpu_helpers import TOL_BF16, bf16_round, normwise_err, say
from oracle import dense, moe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,d,F,E,k,act", [
    (1, 2, 2, 1, 1, "gelu"),        # one input pair, one column
    (3, 30, 34, 3, 2, "relu"),      # chunks of 8 inputs with tails, columns off 32
    (17, 66, 530, 7, 3, "gelu"),    # two and more row tiles, a contraction of many rounds of the ring
    (40, 520, 72, 2, 1, "sigmoid"),  # a long up contraction
    (640, 36, 1030, 64, 2, "gelu"),  # the largest row count, empty and many experts
    (320, 64, 300, 5, 4, "none"),
])
def test_layer(N, d, F, E, k, act):
    import yggdrasil_amd

    g = np.random.default_rng(N + F)
    x = bf16_round(g.standard_normal((N, d, 8)).astype(np.float32))
    lg = g.standard_normal((N, E)).astype(np.float32)
    lg[:, 0] -= 20.0 * (E > k)  # an expert without rows
    wu = bf16_round((g.standard_normal((E, F, d, 8)) / np.sqrt(8 * d)).astype(np.float32))
    wd = bf16_round((g.standard_normal((E, d, F, 8)) / np.sqrt(8 * F)).astype(np.float32))
    bu, bd = ((0.1 * g.standard_normal(s)).astype(np.float32) for s in ((E, F, 8), (E, d, 8)))
    res = bf16_round(g.standard_normal((N, d, 8)).astype(np.float32))
    say(f"few rows N={N} d={d} F={F} E={E} k={k} {act}")
    xt, lt, rt = torch.from_numpy(x).cuda().bfloat16(), torch.from_numpy(lg).cuda(), torch.from_numpy(res).cuda().bfloat16()
    if act == "none":  # the operator takes it, a layer's configuration does not
        from yggdrasil_amd import ops

        wt = [ops.prepare_weights(torch.from_numpy(v).cuda(), "pauli") for v in (wu, wd)]
        bt = [ops.prepare_bias(torch.from_numpy(v).cuda()) for v in (bu, bd)]
        out, routing = ops.moe_forward(xt, k, wt[0], wt[1], bt[0], bt[1], act, logits=lt, residual=rt)
    else:
        cfg = yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=F, n_experts=E, top_k=k, activation=act, dtype=torch.bfloat16,
                                         weight_format="pauli", router="logits")
        layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
        layer.load_reference_weights(w_up=wu, b_up=bu, w_down=wd, b_down=bd)
        out = layer.moe_forward(xt[None], logits=lt, residual=rt[None])[0]
        routing = layer.last_routing
    idx = routing["topk_idx"].cpu().numpy()
    w = routing["topk_w"].cpu().numpy()
    ref = dense.moe_layer(x, idx, w, wu, bu, wd, bd, act, residual=res)
    assert normwise_err(out.float().cpu().numpy(), ref) < TOL_BF16


@pytest.mark.parametrize("E,k", [(1, 1), (7, 2), (33, 4), (64, 3)])
@pytest.mark.parametrize("N", [1, 9, 90, 91, 128, 129, 300, 301, 1024])
def test_route_paths_agree(N, E, k):
    """The same routing on the one- and the two-launch path, from logits and from x (whose logits the one-
    workgroup kernel and the separate launch sum in one order), against the oracle's selection."""
    from yggdrasil_amd import ops

    g = np.random.default_rng(N * E)
    lg = g.standard_normal((N, E)).astype(np.float32)
    say(f"route N={N} E={E} k={k}")
    r = ops.route(torch.from_numpy(lg).cuda(), k)
    idx, w = moe.route_topk(moe.softmax(lg), k)
    counts, offsets, perm, slot_pos = moe.dispatch_plan(idx, E)
    for got, want in ((r.topk_idx, idx), (r.counts, counts), (r.offsets, offsets), (r.perm, perm), (r.slot_pos, slot_pos)):
        assert np.array_equal(got.cpu().numpy().reshape(want.shape), want)
    for dt in (torch.float32, torch.bfloat16):
        for d in (13, 64, 70):
            x = torch.from_numpy(g.standard_normal((N, d, 8)).astype(np.float32)).cuda().to(dt)
            rw, rb = torch.randn(E, 4).cuda(), torch.randn(E).cuda()
            a = ops.route_energy(x, rw, rb, k)
            one = ops.route_energy(x[:1].contiguous(), rw, rb, k)  # one token: always the one-workgroup kernel
            assert torch.equal(a.topk_idx[0], one.topk_idx[0]) and torch.equal(a.topk_w[0], one.topk_w[0])
            sep = ops.route(ops.router_energy_logits(x, rw, rb), k)
            assert (a.topk_idx != sep.topk_idx).float().mean().item() < 0.02  # another order of the sums: ties only


@pytest.mark.parametrize("E,d_in,d_out,counts", [
    (3, 33, 40, (0, 5, 1)),          # a row split over more waves than rows, an empty expert
    (8, 64, 256, (120, 3, 0, 64, 65, 63, 130, 67)),
    (2, 20, 30, (400, 1000)),        # several chunks per expert
    (70, 9, 17, tuple(range(70))),   # more experts than lanes
])
def test_weight_gradient_row_split(E, d_in, d_out, counts):
    """The weight gradient of few rows: each expert against float64 (sums of up to 1000 rows x 4 terms in fp32:
    2^-24 sqrt(4000) of a random sum; 1e-5)."""
    from yggdrasil_amd import ops

    g = np.random.default_rng(E + d_in)
    P = sum(counts)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    a, dy = (g.standard_normal((P, n, 8)).astype(np.float32) for n in (d_in, d_out))
    say(f"weight gradient E={E} {d_in} x {d_out}")
    dW, db = ops.grouped_weight_grad_pauli(ops.pauli_rows_from_blade_f32(torch.from_numpy(dy).cuda()),
                                           ops.pauli_rows_from_blade_f32(torch.from_numpy(a).cuda()),
                                           torch.from_numpy(off).cuda(), E)
    for e in range(E):
        _, want, want_b = dense.linear_backward(a[off[e]:off[e + 1]], np.zeros((d_out, d_in, 8)), dy[off[e]:off[e + 1]])
        if counts[e] == 0:
            assert not dW[e].any() and not db[e].any()
        else:
            assert normwise_err(dW[e].cpu().numpy(), want) < 1e-5 and normwise_err(db[e].cpu().numpy(), want_b) < 1e-5


def test_adjoint_preparation_and_balance_loss():
    """One-pass adjoint weights equal the two-pass ones bit for bit; the balance loss is the formula's."""
    from yggdrasil_amd import ops

    w = torch.randn(3, 37, 50, 8, device="cuda")
    assert torch.equal(ops.prepare_adjoint_weights(w).data, ops.prepare_weights(ops.adjoint_weights(w), "pauli_f32").data)
    for E in (1, 8, 64, 100):
        c = torch.randint(0, 3000, (E,), device="cuda", dtype=torch.int32)
        f = c.double() / (c.double().sum() + 1e-12)
        assert abs(ops.balance_loss(c).item() - ((f - 1.0 / E) ** 2).sum().item()) <= 1e-6 * max(1.0 / E, 1e-3)
    assert ops.balance_loss(torch.zeros(8, device="cuda", dtype=torch.int32)).item() == pytest.approx(1.0 / 8)


@pytest.mark.parametrize("N,d,F,E,k,act", [
    (200, 17, 18, 3, 2, "gelu"),     # two chunks of the contraction, the second one input long; odd width
    (333, 101, 131, 5, 2, "sigmoid"),  # odd widths, columns off 64 and 32
    (900, 64, 129, 4, 1, "relu"),    # odd hidden width (a padding column between the products)
    (160, 150, 70, 2, 2, "gelu"),
])
def test_int8_layer_of_enough_rows(N, d, F, E, k, act):
    """int8 weights: the layer on the dequantized weights (x and weights exact; h, y and the output rounded to bf16),
    tokens over many binades, an expert without rows, a token of zeros."""
    import yggdrasil_amd

    g = np.random.default_rng(N + F)
    x = g.standard_normal((N, d, 8)).astype(np.float32) * np.ldexp(1.0, g.integers(-12, 5, (N, 1, 1))).astype(np.float32)
    x[5] = 0.0
    x = bf16_round(x)
    lg = g.standard_normal((N, E)).astype(np.float32)
    lg[:, 0] -= 30.0 * (E > k)
    wu = (g.standard_normal((E, F, d, 8)) / np.sqrt(8 * d)).astype(np.float32)
    wd = (g.standard_normal((E, d, F, 8)) / np.sqrt(8 * F)).astype(np.float32)
    bu, bd = ((0.1 * g.standard_normal(s)).astype(np.float32) for s in ((E, F, 8), (E, d, 8)))
    cfg = yggdrasil_amd.MoEHLMConfig(d_model=d, d_ff=F, n_experts=E, top_k=k, activation=act, dtype=torch.bfloat16,
                                     weight_format="int8", router="logits")
    layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
    layer.load_reference_weights(w_up=wu, b_up=bu, w_down=wd, b_down=bd)
    say(f"int8 layer N={N} d={d} F={F} E={E} k={k} {act}")
    out = layer.moe_forward(torch.from_numpy(x).cuda().bfloat16()[None], logits=torch.from_numpy(lg).cuda())[0]
    idx = layer.last_routing["topk_idx"].cpu().numpy()
    w = layer.last_routing["topk_w"].cpu().numpy()
    ref = dense.moe_layer(x, idx, w, moe.dequantize_int8(*moe.quantize_int8(wu)), bu,
                          moe.dequantize_int8(*moe.quantize_int8(wd)), bd, act)
    got = out.float().cpu().numpy()
    # y and the output are rounded once each, 2^-9 of an element at most, and k rows of y are added
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2.0 ** -8
    assert normwise_err(got, ref) < TOL_BF16


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layer_with_pruned_and_parametrized_weights(dtype):
    """A pruned weight is no parameter of that name any more, a parametrized one lies in a submodule: same outputs, bit
    for bit, and a change of the tensor behind it is seen."""
    import copy

    import torch.nn.utils.parametrize as parametrize
    import torch.nn.utils.prune as prune
    import yggdrasil_amd

    cfg = yggdrasil_amd.MoEHLMConfig(d_model=32, d_ff=64, n_experts=4, top_k=2, dtype=dtype)
    layer = yggdrasil_amd.CliffordMoELayer(cfg, device="cuda")
    other = copy.deepcopy(layer)
    prune.identity(other, "w_up")
    prune.identity(other, "router_weight")
    parametrize.register_parametrization(other, "b_down", torch.nn.Identity())
    x = torch.randn(1, 40, 32, 8, device="cuda").to(dtype)
    with torch.no_grad():
        assert torch.equal(layer.moe_forward(x), other.moe_forward(x))
        layer.b_down.add_(1.0)
        other.parametrizations.b_down.original.add_(1.0)
        assert torch.equal(layer.moe_forward(x), other.moe_forward(x))
