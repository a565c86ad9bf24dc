"""The per-token expert kernels at the widths where their units run out: rows of one block, of 63 to 65
blocks (64 lanes, one block each), and activations up to and past the size where the padding of their
blocks no longer fits. Reference: f64 on the dequantized weights; bar 1e-5 of a token's largest output
(f32 products and sums of up to 4,096 terms in 64 lanes: some 1e-6)."""
import npref
import numpy as np
import pytest

import moe_rocm as M
from moe_rocm import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ggml_type,H,I,sh", [
    (W.GGML_MXFP4, 32, 32, 0), (W.GGML_MXFP4, 2016, 96, 0), (W.GGML_MXFP4, 2048, 64, 32), (W.GGML_MXFP4, 256, 64, 256), (W.GGML_MXFP4, 2080, 2080, 0),
    (W.GGML_MXFP4, 64, 3616, 96), (W.GGML_MXFP4, 64, 3648, 0), (W.GGML_Q4_K, 256, 256, 0), (W.GGML_Q4_K, 2304, 256, 512),
    (W.GGML_Q4_K, 256, 3584, 256), (W.GGML_Q4_K, 256, 3584, 0)])
def test_valu_widths(gpu_ctx, ggml_type, H, I, sh):
    spec = W.LayerSpec(282, 0, ggml_type, H, I, 5, 4, W.ROUTE_NORM_TOPK, W.ACT_SILU, ggml_type == W.GGML_MXFP4,
                       True, sh_inter=sh, sh_type=W.GGML_Q4_K if sh % 256 == 0 else W.GGML_MXFP4)
    host = W.host_layer(spec)
    dl = W.DeviceLayer(gpu_ctx, spec, host=host)
    T = 3
    x = W.x_tokens(spec, T)
    dx, dy = gpu_ctx.to_device(x), gpu_ctx.alloc(T * H * 4)
    gpu_ctx.set_option(M.OPT_DECODE_KERNEL, M.DECODE_VALU)
    try:
        dl.layer.forward_batched(dx, T, dy)
        gpu_ctx.sync()
        got = dy.download(np.float32).reshape(T, H)
        ref = npref.moe_forward(host, x)[0]
        assert (np.abs(got - ref).max(1) <= 1e-5 * np.abs(ref).max(1)).all()
    finally:
        gpu_ctx.set_option(M.OPT_DECODE_KERNEL, M.DECODE_AUTO)
        dx.free(), dy.free()
        dl.close()
