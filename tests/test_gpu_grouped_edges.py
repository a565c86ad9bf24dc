"""The grouped multi-token kernels at the edges of their tiles: pair counts around the 16-, 32- and
64-pair tiles and their 16-pair groups (all tokens on the same experts, so an expert's pairs are
the tokens), calls that select each pair tile and row count per work item, one and several super-blocks per row, row counts
that fill half a tile, the shared expert's own width, and enough pairs for the grouping to take
several workgroups. Reference: the per-token VALU path (f32 arithmetic, 3e-7 of the output), per
token, max error over the token's largest output. Bar 2e-5 for Q4_K: the activations carry 22
significant bits and sums are f32."""
from dataclasses import replace

import numpy as np
import pytest

import moe_rocm as M
from moe_rocm import workloads as W

pytestmark = pytest.mark.gpu

Q4 = W.LayerSpec(280, 0, W.GGML_Q4_K, 512, 256, 24, 3, W.ROUTE_NORM_TOPK, W.ACT_SILU, False, True)
BAR = 2e-5


def _batched(gpu_ctx, dl, x, kernel):
    T, H = x.shape
    dx, dy = gpu_ctx.to_device(x), gpu_ctx.alloc(T * H * 4)
    gpu_ctx.set_option(M.OPT_DECODE_KERNEL, kernel)
    try:
        dl.layer.forward_batched(dx, T, dy)
        gpu_ctx.sync()
        return dy.download(np.float32).reshape(T, H)
    finally:
        gpu_ctx.set_option(M.OPT_DECODE_KERNEL, M.DECODE_AUTO)
        dx.free(), dy.free()


def _one_route(host, spec):
    """The router bias decides: every token takes the same top_k experts."""
    host["router_b"] = (host["router_b"] + 1e3 * (np.arange(spec.n_experts) % 5 == 1)
                        - np.arange(spec.n_experts)).astype(np.float32)
    return host


def _check_layer(gpu_ctx, dl, T, bar=BAR):
    x = W.x_tokens(dl.spec, T)
    ref = _batched(gpu_ctx, dl, x, M.DECODE_VALU)
    got = _batched(gpu_ctx, dl, x, M.DECODE_AUTO)
    err = np.abs(got - ref).max(1) / np.abs(ref).max(1)
    assert np.isfinite(got).all() and err.max() <= bar, (dl.spec, T, float(err.max()), int(err.argmax()))


def _check(gpu_ctx, spec, T, one_route=False, bar=BAR):
    host = W.host_layer(spec)
    dl = W.DeviceLayer(gpu_ctx, spec, host=_one_route(host, spec) if one_route else host)
    try:
        _check_layer(gpu_ctx, dl, T, bar)
    finally:
        dl.close()


@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 31, 33, 48, 49, 63, 64, 65, 129])
def test_q4k_pairs_per_expert(gpu_ctx, T):
    _check(gpu_ctx, Q4, T, one_route=True)


@pytest.mark.parametrize("T", [64, 65])  # 8 pairs per expert in the mean and just above
def test_q4k_pair_tile_rule(gpu_ctx, T):
    _check(gpu_ctx, Q4, T)


# 10 super-blocks of 256 gate rows, 3 super-blocks per gate/up row and 10 per down row; every token on the same
# three of 12 experts. Gate/up items of 64 rows up to 37 tokens, of 128 rows up to 149 (16-pair tiles both),
# then 64-pair tiles of 256 rows, whose last tile holds 1, 2, 3 or 4 16-pair groups.
WIDE = replace(Q4, hidden=768, inter=2560, n_experts=12)


@pytest.fixture(scope="module", params=[0, 256], ids=["routed", "shared"])
def wide_layer(gpu_ctx, request):
    spec = replace(WIDE, sh_inter=request.param)
    dl = W.DeviceLayer(gpu_ctx, spec, host=_one_route(W.host_layer(spec), spec))
    yield dl
    dl.close()


@pytest.mark.parametrize("T", [1, 15, 16, 17, 33, 37, 38, 47, 48, 49, 64, 65, 149, 160, 161, 176, 177, 191, 192, 193,
                               207, 208, 209])
def test_q4k_work_items(gpu_ctx, wide_layer, T):
    _check_layer(gpu_ctx, wide_layer, T)


def test_q4k_sub_block_sums(gpu_ctx):
    """A down matrix of minimums alone: row 8 b + j is minus the sum of h over sub-block j of super-block b.
    Each sum goes to the down kernel as three f16 terms, which several lanes write: some 300,000 sums, so that
    many lie where two lanes' roundings of the same sum could part (2^-11 of it then, fifty times the bar)."""
    H, nsb, E = WIDE.hidden, WIDE.inter // 256, WIDE.n_experts
    host = W.host_layer(WIDE)
    down = np.zeros((E, H, nsb, 144), np.uint8)
    for b in range(nsb):
        for j in range(8):
            down[:, 8 * b + j, b, 2:4] = np.frombuffer(np.float16(1).tobytes(), np.uint8)  # dmin
            down[:, 8 * b + j, b, 8 + j] = 1 if j < 4 else 16  # m_j = 1
    host["down"] = down.reshape(-1)
    dl = W.DeviceLayer(gpu_ctx, WIDE, host=host)
    try:
        for T in (30, 60, 1400):  # each kind of work item
            _check_layer(gpu_ctx, dl, T)
    finally:
        dl.close()


def _ran(gpu_ctx, dl, T, scope):
    """Launches named `scope` in a batched call of T tokens."""
    gpu_ctx.profile_reset()
    gpu_ctx.set_option(M.OPT_PROFILE, 1)
    try:
        _batched(gpu_ctx, dl, W.x_tokens(dl.spec, T), M.DECODE_AUTO)
        return gpu_ctx.profile_read(scope)[0]
    finally:
        gpu_ctx.set_option(M.OPT_PROFILE, 0)


# Few tokens, and many tokens of few narrow experts: 24 and 16 items of 256 rows, or 24 of 64 pairs and 256
# rows, leave nine in ten CUs idle (28, 31 and 81% slower than smaller items). Smaller items pass h through
# memory (split_h); with an item for every second CU they need not be smaller.
@pytest.mark.parametrize("E,k,H,I,T,small", [(128, 8, 2048, 768, 1, True), (16, 2, 2048, 256, 8, True),
                                             (16, 2, 2048, 256, 512, True), (12, 3, 768, 2560, 160, False)])
def test_q4k_few_work_items_are_split(gpu_ctx, E, k, H, I, T, small):
    spec = replace(Q4, hidden=H, inter=I, n_experts=E, top_k=k)
    dl = W.DeviceLayer(gpu_ctx, spec)
    try:
        assert _ran(gpu_ctx, dl, T, "split_h") == (1 if small else 0)
    finally:
        dl.close()


@pytest.mark.parametrize("H,I,sh", [(256, 256, 0), (768, 512, 256), (1280, 768, 1024), (2048, 256, 512)])
@pytest.mark.parametrize("T", [5, 70])
def test_q4k_widths_and_shared(gpu_ctx, H, I, sh, T):
    _check(gpu_ctx, replace(Q4, hidden=H, inter=I, sh_inter=sh), T)


# MXFP4: the activations carry three 8-bit float terms; what they leave is below 2^-12 of a block's
# largest value in each of the two products.
MX = W.LayerSpec(281, 0, W.GGML_MXFP4, 288, 2080, 24, 3, W.ROUTE_SOFTMAX_AFTER_TOPK, W.ACT_SWIGLU_OAI, True, True)
MX_BAR = 2.0 ** -11


# 17 row tiles of the 2,080 gate rows (the last of 32 rows), 9 blocks per row of 288; every token on the
# same three experts. 16-pair tiles up to 96 tokens (a mean of 12 pairs per expert), then 32-pair tiles; the
# counts leave the last tile around each edge of its 16-pair groups.
@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 33, 64, 65, 80, 81, 96, 97, 256, 683, 704, 705, 720, 721, 735, 737,
                               753])
def test_mxfp4_pairs_per_expert(gpu_ctx, T):
    _check(gpu_ctx, MX, T, one_route=True, bar=MX_BAR)


# Two of six experts, 33 blocks per row: from about 1,900 tokens on 64-pair tiles, two rounds of work items.
# The last tile around each edge of its 16-pair groups.
@pytest.mark.parametrize("T", [1985, 2000, 2001, 2016, 2017, 2032, 2033, 2047, 2048])
def test_mxfp4_64_pair_tiles(gpu_ctx, T):
    _check(gpu_ctx, replace(MX, hidden=1056, n_experts=6, top_k=2), T, one_route=True, bar=MX_BAR)


@pytest.mark.parametrize("H,I,sh", [(32, 32, 0), (160, 96, 0), (1056, 288, 2080), (2880, 160, 64)])
@pytest.mark.parametrize("T", [5, 150, 1100])  # 1,100 tokens x 17 row tiles: the shared expert in 32-pair tiles
def test_mxfp4_widths_and_shared(gpu_ctx, H, I, sh, T):
    _check(gpu_ctx, replace(MX, hidden=H, inter=I, sh_inter=sh, sh_type=W.GGML_MXFP4), T, bar=MX_BAR)


@pytest.mark.parametrize("spec", [replace(MX, hidden=1056, inter=288), replace(Q4, hidden=768, sh_inter=512),
                                  replace(MX, hidden=160, inter=96, sh_inter=64, sh_type=W.GGML_MXFP4)])
@pytest.mark.parametrize("kernel", [M.DECODE_AUTO, M.DECODE_VALU])
@pytest.mark.parametrize("T", [2, 33])
def test_residual_added_in_the_combine(gpu_ctx, spec, kernel, T):
    """h + moe(norm(h)) is the plain call's result on the normed rows plus h, and the same bits
    into another buffer and in place."""
    dl = W.DeviceLayer(gpu_ctx, spec, host=W.host_layer(spec))
    h = W.x_tokens(spec, T) * np.float32(2.0) ** -3
    one = np.ones(spec.hidden, np.float32)
    zero = np.zeros_like(h)
    dh, dn, dy, dz = (gpu_ctx.to_device(v) for v in (h, one, zero, zero))
    gpu_ctx.set_option(M.OPT_DECODE_KERNEL, kernel)
    try:
        dl.layer.forward_batched_residual(dh, T, dn, 1e-5, dy)
        dl.layer.forward_batched_residual(dh, T, dn, 1e-5, dh)
        gpu_ctx.sync()
        out, in_place = dy.download(np.float32), dh.download(np.float32)
        assert np.array_equal(out, in_place)
        normed = (h * (np.float32(1) / np.sqrt((h.astype(np.float64) ** 2).mean(1, keepdims=True) + 1e-5))).astype(np.float32)
        dx = gpu_ctx.to_device(normed)
        dl.layer.forward_batched(dx, T, dz)
        gpu_ctx.sync()
        want = h + dz.download(np.float32).reshape(h.shape)
        # the norm's own rounding (a few 2^-24 of its sum of squares) passes through the layer
        assert np.abs(out.reshape(h.shape) - want).max() <= MX_BAR * np.abs(want).max()
        dx.free()
    finally:
        gpu_ctx.set_option(M.OPT_DECODE_KERNEL, M.DECODE_AUTO)
        for b in (dh, dn, dy, dz):
            b.free()
        dl.close()


@pytest.mark.parametrize("T", [2730, 2731, 5500])  # 8,190, 8,193 and 16,500 pairs: one, two and three workgroups
def test_grouping_of_many_pairs(gpu_ctx, T):
    _check(gpu_ctx, replace(Q4, hidden=256), T)


def test_q4k_scales_zero_and_denormal_rows(gpu_ctx):
    """Rows of zeros, of denormals, of 2^100 and of mixed magnitudes: the power-of-two row scale."""
    spec = replace(Q4, hidden=512)
    host = W.host_layer(spec)
    host["router_w"] = np.zeros_like(host["router_w"])
    dl = W.DeviceLayer(gpu_ctx, spec, host=host)
    try:
        x = W.x_tokens(spec, 20)
        x[0] = 0.0
        x[1] = 1e-40
        x[2] *= np.float32(1e-30)
        x[3] *= np.float32(2.0) ** 40
        x[4, ::2] *= np.float32(1e-6)
        ref = _batched(gpu_ctx, dl, x, M.DECODE_VALU)
        got = _batched(gpu_ctx, dl, x, M.DECODE_AUTO)
        assert np.array_equal(got[0], ref[0]) and np.abs(got[1]).max() <= 1e-30
        for t in range(2, 20):
            assert np.abs(got[t] - ref[t]).max() <= BAR * np.abs(ref[t]).max() + 1e-37, t
    finally:
        dl.close()


def test_q4k_call_in_parts(gpu_ctx):
    """More tokens than the images' 31-bit offsets cover (30,599 of hidden size 16,384) run in parts: every
    token's result is that of the same row in a small call, without and with the residual, in place."""
    H, n = 16384, 601
    T = 0x7F000000 // (H // 256 * 1088) + 37
    spec = replace(Q4, hidden=H, n_experts=7, top_k=2, sh_inter=256)
    ctx = M.Context(0)  # its scratch goes with it
    dl = W.DeviceLayer(ctx, spec, host=_one_route(W.host_layer(spec), spec))
    try:
        base = W.x_tokens(spec, n)
        norm_w = ctx.to_device(W.norm_weights(1, H)[0])
        dx = ctx.to_device(base)
        want = ctx.alloc(n * H * 4)
        dl.layer.forward_batched(dx, n, want)
        dl.layer.forward_batched_residual(dx, n, norm_w, 1e-5, dx)
        ctx.sync()
        plain, resid = (b.download(np.float32).reshape(n, H) for b in (want, dx))
        dx.free(), want.free()
        rows = np.arange(T) % n
        dx, dy = ctx.to_device(base[rows]), ctx.alloc(T * H * 4)
        dl.layer.forward_batched(dx, T, dy)
        dl.layer.forward_batched_residual(dx, T, norm_w, 1e-5, dx)
        ctx.sync()
        for buf, ref in ((dy, plain), (dx, resid)):
            got = buf.download(np.float32).reshape(T, H)
            for t0 in range(0, T, n):  # block by block: the whole is 2 GB
                g = got[t0:t0 + n]
                r = ref[:g.shape[0]]
                assert (np.abs(g - r).max(1) <= BAR * np.abs(r).max(1)).all(), t0
        for b in (dx, dy, norm_w):
            b.free()
    finally:
        dl.close()
        ctx.close()
