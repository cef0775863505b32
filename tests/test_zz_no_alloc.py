"""ohip_conv2d_noalloc (no device allocation, static per-GPU scratch) against
ohip_conv2d through the C ABI: identical results on two calls in a row, the
second with a smaller input, and no device allocation by either noalloc
call.  The cases use the scratch: an NCHW input (the staging copy) and a
split-K contraction (partial sums)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a GPU"
    return t


@pytest.fixture(scope="module")
def ctx(torch):
    from oxionnx_amd.device import HipContext
    c = HipContext(0)
    yield c
    c.close()


def _case(torch, ctx, dt, xs, ws, pads, seed):
    from oxionnx_amd import _lib as L
    rng = np.random.default_rng(seed)
    tdt = {"f32": torch.float32, "f16": torch.float16}[dt]
    x = torch.from_numpy(rng.uniform(-1, 1, xs).astype(np.float32)).cuda().to(tdt)
    w = rng.normal(0, 0.05, ws).astype(np.float32)
    b = torch.from_numpy(rng.normal(0, 0.01, ws[0]).astype(np.float32)).cuda().to(tdt)
    wt = ctx.weight_conv(w, dtype=L.F32 if dt == "f32" else L.F16)
    return x, wt, b


# (dtype, x shape, w shape, pads, strides).  Every call uses the scratch:
# the f16 calls stage their NCHW input as NHWC (the first also splits K on
# the halo-patch path, a 512 -> 512 3x3 conv at 32x32, 4.8 GFLOP); the f32
# 512 -> 512 conv takes the halo-patch path too (staging + split-K partial
# sums: the f32 NCHW kernel that reads its input in place is used only
# below the halo path's 3 GFLOP), and the second f32 call has stride 2,
# which that in-place kernel does not take, so it stages its input for the
# engine
CALLS = [("f16", (1, 512, 32, 32), (512, 512, 3, 3), (1, 1, 1, 1), (1, 1)),
         ("f16", (1, 64, 20, 24), (96, 64, 3, 3), (1, 1, 1, 1), (1, 1)),
         ("f32", (1, 512, 32, 32), (512, 512, 3, 3), (1, 1, 1, 1), (1, 1)),
         ("f32", (2, 16, 9, 11), (24, 16, 3, 3), (0, 1, 2, 1), (2, 2))]


@pytest.mark.parametrize("pair", [(0, 1), (2, 3)], ids=["f16", "f32"])
def test_noalloc_matches_conv2d_twice(torch, ctx, pair):
    from oxionnx_amd import _lib as L
    for i in pair:
        dt, xs, ws, pads, strides = CALLS[i]
        x, wt, b = _case(torch, ctx, dt, xs, ws, pads, seed=i)
        want = ctx.conv2d(x, wt, b, strides=strides, pads=pads, act=L.ACT_RELU)
        got = torch.full_like(want, float("nan"))
        torch.cuda.synchronize()
        ctx.reset_counters()
        ctx.conv2d(x, wt, b, strides=strides, pads=pads, act=L.ACT_RELU, out=got, noalloc=True)
        torch.cuda.synchronize()
        assert ctx.counters()["device_allocs"] == 0
        assert torch.equal(got, want), (i, float((got.float() - want.float()).abs().max()))


def test_noalloc_rejects_more_scratch_than_the_static_array(torch, ctx):
    from oxionnx_amd import _lib as L
    # an NCHW f16 input of 40 MiB needs an NHWC staging copy larger than
    # 32 MiB (f32 NCHW 1x1 / 3x3 convs read their input in place)
    x = torch.zeros((1, 320, 256, 256), dtype=torch.float16, device="cuda")
    wt = ctx.weight_conv(np.zeros((16, 320, 1, 1), np.float32), dtype=L.F16)
    out = torch.zeros((1, 16, 256, 256), dtype=torch.float16, device="cuda")
    with pytest.raises(L.OhipError) as e:
        ctx.conv2d(x, wt, None, out=out, noalloc=True)
    assert e.value.code == L.E_NOMEM and "static" in str(e.value)


# a halo-path f32 convolution whose K slices, or whose staged input, exceed
# 32 MiB: unsplit, or in place (whole numbers: the same sums in any order)
@pytest.mark.parametrize("xs,cout", [((1, 192, 128, 128), 192), ((9, 64, 128, 128), 64)], ids=["slices", "staging"])
def test_noalloc_halo_without_room(torch, ctx, xs, cout):
    rng = np.random.default_rng(xs[1])
    x = torch.from_numpy(rng.integers(-3, 4, xs).astype(np.float32)).cuda()
    wt = ctx.weight_conv(rng.integers(-3, 4, (cout, xs[1], 3, 3)).astype(np.float32))
    want = ctx.conv2d(x, wt, pads=(1, 1, 1, 1))
    got = torch.full_like(want, float("nan"))
    torch.cuda.synchronize()
    ctx.reset_counters()
    ctx.conv2d(x, wt, pads=(1, 1, 1, 1), out=got, noalloc=True)
    torch.cuda.synchronize()
    assert ctx.counters()["device_allocs"] == 0
    assert torch.equal(got, want)


# an image of 2 GiB, past the in-place f32 kernel's 31-bit offsets: the same
# sums as the bands of rows that it is cut into here, and no staged copy
@pytest.mark.parametrize("k,mode", [(3, "zeros"), (1, "zeros"), (3, "reflect")])
def test_noalloc_of_an_image_past_31_bits(torch, ctx, k, mode):
    from oxionnx_amd import _lib as L
    c, cout, h, w = 64, 12, 2900, 2901
    x = torch.empty((1, c, h, w), device="cuda")
    x.uniform_(-1, 1, generator=torch.Generator(device="cuda").manual_seed(k))
    rng = np.random.default_rng(k)
    wt = ctx.weight_conv(rng.normal(0, 0.1, (cout, c, k, k)).astype(np.float32))
    p = k // 2
    y = torch.full((1, cout, h, w), float("nan"), device="cuda")

    def call(src, dst, rows, pt, pb):   # (the descriptor takes the pad mode, which conv2d() does not)
        d = L.ConvDesc(1, c, rows, w, cout, k, k, 1, 1, 1, 1, 1, pt, p, pb, p, L.F32, L.NCHW, L.NCHW, L.ACT_NONE, 0.0, 0.0,
                       L.PAD_REFLECT if mode == "reflect" else L.PAD_ZEROS)
        L.check(L.lib().ohip_conv2d_noalloc(ctx.h, ctypes.byref(d), src.data_ptr(), wt.handle, None, dst.data_ptr()))

    torch.cuda.synchronize()
    ctx.reset_counters()
    call(x, y, h, p, p)
    torch.cuda.synchronize()
    assert ctx.counters()["device_allocs"] == 0
    for r0, r1 in ((0, 64), (1400, 1464), (h - 64, h)):   # output rows; the bands' inner edges have no pad
        a, b = max(r0 - p, 0), min(r1 + p, h)
        pt, pb = (p if a == 0 else 0), (p if b == h else 0)
        part = torch.empty((1, cout, b - a + pt + pb - 2 * p, w), device="cuda")
        call(x[:, :, a:b].contiguous(), part, b - a, pt, pb)
        assert torch.equal(y[:, :, r0:r1], part)
    assert not bool(torch.isnan(y).any())
