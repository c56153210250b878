"""The position-major Vocos stages (qtts_dconv.hip) where their tiles end:
lengths from one position up, each tile form (256, 128 and 64 positions, the
contraction over waves and over slices), one and several channel tiles,
kernel = stride and 2 stride, every dilation, a block without residuals.

Against the float64 decoder.  A convolution of n products is an f32 sum of
3n / 32 roundings at most (one per matrix instruction) of operands within
2^-22 of their own f32: relative to its terms' sum 2^-22 + 3n / 32 2^-24, that
is 4e-6 at the 672 products of a 96-channel k 7 convolution; about eight of
them follow each other here, at unit gain: 3.2e-5 of the signal.
"""
import numpy as np
import pytest

import f64decoder as F
from qtts import synth

pytestmark = pytest.mark.gpu
TOL = 3.2e-5


def decoder(vocos, rates, dilations=(1, 3, 9), latent=64, **kw):
    return synth.make_decoder(seed=61, latent=latent, hidden=64, n_heads=4, head_dim=16, inter=128, n_tf_layers=1,
                              codebook_size=64, codebook_dim=32, vq_dim=32, vocos=vocos, rates=rates,
                              dilations=dilations, rope_max_pos=4096, **kw)


def run(ctx, d, frames):
    ctx.upload_decoder(d)
    assert ctx.debug_query("decoder_rows") == 2      # (heads of 16: the transformer stays channel-first)
    rng = np.random.Generator(np.random.PCG64(frames))
    for T in frames if isinstance(frames, tuple) else (frames,):
        print(f"frames {T}", flush=True)
        codes = rng.integers(0, 64, (16, T)).astype(np.uint32)
        ref = F.decode(d, codes)
        got = ctx.decode_to_audio(codes)
        assert got.shape == ref.shape
        assert ctx.debug_query("decode_repeated") == 0
        err = np.abs(got.astype(np.float64) - ref).max() / np.abs(ref).max()
        assert err <= TOL, f"{T} frames: {err:.3g} of the largest sample"


@pytest.fixture(scope="module")
def ctx(ctx_factory):
    return ctx_factory(64)


def test_one_channel_tile(ctx):
    """96 channels throughout (the residual units as one launch), 4 x 3
    positions a frame and more: 12 to 8,412 positions."""
    run(ctx, decoder((96, 96), (3,)), (1, 2, 5, 6, 21, 22, 43, 701))


def test_several_channel_tiles(ctx):
    run(ctx, decoder((288, 192, 96), (5, 2)), (1, 3, 13, 26, 107, 240))


def test_wide_contraction(ctx):
    """Many records and few positions: slices of the contraction.  (192
    channels at the end: the output convolution's tile holds no more than 208,
    and a decoder beyond that stays channel-first.)"""
    run(ctx, decoder((768, 384, 192), (4, 2), latent=256), (1, 4, 33))


def test_no_residuals(ctx):
    run(ctx, decoder((96, 192), (2,), dilations=()), (1, 17, 90))


def test_stride_kernel(ctx):
    """Transposed convolutions of kernel = stride: one tap."""
    d = decoder((96, 96), (4,))
    c = d.vocos_blocks[0].upsample
    c.weight, c.kernel_size = np.ascontiguousarray(c.weight[:, :, :4]), 4
    run(ctx, d, (1, 9, 130))


def test_quiet_channels_beside_loud_ones(ctx, monkeypatch):
    """One 96-channel tile of the first signal near 1e-7 (below what lo
    carries) beside a loud one: the range check looks at all channels of the
    positions, so the decode stays on the split path (other bits than the f32
    one's), and is as accurate."""
    d = decoder((192, 96), (3,))
    c = d.vocos_init
    c.weight[:96] *= np.float32(1e-7)
    c.bias[:96] *= np.float32(1e-7)
    run(ctx, d, (1, 40, 150))
    codes = np.random.Generator(np.random.PCG64(5)).integers(0, 64, (16, 40)).astype(np.uint32)
    got = ctx.decode_to_audio(codes)
    monkeypatch.setenv("QTTS_DEC_F32", "1")
    assert not np.array_equal(got.view(np.uint32), ctx.decode_to_audio(codes).view(np.uint32))


def scaled(a, f):
    a *= np.float32(f)


@pytest.mark.parametrize("case", ["quiet", "loud"])
def test_out_of_range_signal_repeats_the_decode(ctx, monkeypatch, case):
    """The first Vocos signal wholly near 1e-6, or past the f16 maximum, behind
    inputs and weights within the range: the decode is repeated on the f32 path
    (its bits)."""
    d = decoder((192, 96), (3,))
    if case == "quiet":
        u = d.upsample[-1]                        # its signal near 1e-3 (and the weights above 2^-14)
        scaled(u.conv_t.weight, 1e-3)
        scaled(u.conv_t.bias, 1e-3)
        scaled(u.gamma, 1e-4)
        scaled(d.vocos_init.weight, 1e-3)
        scaled(d.vocos_init.bias, 1e-7)
    else:
        scaled(d.vocos_init.weight, 6e4)
    ctx.upload_decoder(d)
    for T in (1, 40, 150):
        codes = np.random.Generator(np.random.PCG64(T)).integers(0, 64, (16, T)).astype(np.uint32)
        monkeypatch.delenv("QTTS_DEC_F32", raising=False)
        got = ctx.decode_to_audio(codes)
        assert ctx.debug_query("decode_repeated") == 1, f"{T} frames"
        monkeypatch.setenv("QTTS_DEC_F32", "1")
        assert np.array_equal(got.view(np.uint32), ctx.decode_to_audio(codes).view(np.uint32)), f"{T} frames"
