"""Cases where the size of one value must not cost another its bits: inputs that cancel, rows and channels
of very different size, gradients of small rows beside large ones."""

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
