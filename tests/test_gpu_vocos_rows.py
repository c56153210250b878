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
    rng = np.random.Generator(np.random.PCG64(frames))
    for T in frames if isinstance(frames, tuple) else (frames,):
        print(f"frames {T}", flush=True)
        codes = rng.integers(0, 64, (16, T)).astype(np.uint32)
        ref = F.decode(d, codes)
        got = ctx.decode_to_audio(codes)
        assert got.shape == ref.shape
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
    """Many records and few positions: slices of the contraction."""
    run(ctx, decoder((768, 384), (4,), latent=256), (1, 4, 33))


def test_no_residuals(ctx):
    run(ctx, decoder((96, 192), (2,), dilations=()), (1, 17, 90))


def test_stride_kernel(ctx):
    """Transposed convolutions of kernel = stride: one tap."""
    d = decoder((96, 96), (4,))
    c = d.vocos_blocks[0].upsample
    c.weight, c.kernel_size = np.ascontiguousarray(c.weight[:, :, :4]), 4
    run(ctx, d, (1, 9, 130))
