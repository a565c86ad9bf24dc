"""Router logits of many tokens where a workgroup takes one 16 x 16 tile or 2 x 2 of them: token and
expert counts around the tiles and around the size where the choice changes, one range of the hidden
size and several. Reference: f64. Bar: an f32 sum of at most 96 products a wave, then 16 waves and 4
ranges, is off by no more than 116 roundings of 2^-24 of the sum of the products' magnitudes."""
from dataclasses import replace

import numpy as np
import pytest

from moe_rocm import workloads as W

pytestmark = pytest.mark.gpu
SPEC = W.LayerSpec(281, 0, W.GGML_MXFP4, 256, 32, 504, 4, W.ROUTE_SOFTMAX_AFTER_TOPK, W.ACT_SILU, True, True)


@pytest.mark.parametrize("T,E,H", [(496, 504, 256), (497, 504, 256), (511, 504, 256), (529, 481, 256), (545, 512, 32),
                                   (1809, 129, 64), (240, 504, 1568), (241, 504, 1568), (270, 490, 1600)])
def test_router_logits_tiles(gpu_ctx, T, E, H):
    spec = replace(SPEC, n_experts=E, hidden=H)
    host = W.host_layer(spec)
    dl = W.DeviceLayer(gpu_ctx, spec, host=host)
    x = W.x_tokens(spec, T)
    dx, lg = gpu_ctx.to_device(x), gpu_ctx.alloc(T * E * 4)
    di, dw = gpu_ctx.alloc(T * 16), gpu_ctx.alloc(T * 16)
    try:
        dl.layer.router_topk(dx, T, di, dw, lg)
        gpu_ctx.sync()
        got = lg.download(np.float32).reshape(T, E)
        wr = host["router_w"].reshape(E, H).astype(np.float64)
        b = host["router_b"].reshape(1, E).astype(np.float64)
        x64 = x.astype(np.float64)
        bar = 118 * 2.0 ** -24 * (np.abs(x64) @ np.abs(wr).T + np.abs(b))
        assert (np.abs(got - (x64 @ wr.T + b)) <= bar).all()
    finally:
        dx.free(), lg.free(), di.free(), dw.free()
        dl.close()
