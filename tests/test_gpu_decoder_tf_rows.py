"""The decoder's position-major transformer (qtts_dconv.hip) where its tiles
end: positions around the 16 of a matrix tile, the 64 of a workgroup and the
attention window, hidden sizes of both norm kernels, a record count that the
waves do not divide, one head and several.

Against the float64 decoder.  A matrix of n inputs is an f32 sum of 3n / 32
roundings at most of operands within 2^-22 of their own f32, relative to its
terms' sum 2^-22 + 3n / 32 2^-24: 3.5e-6 at 576.  Two layers and the two
projections are ten of them in turn, 3.5e-5; the Vocos stages after them add
eight of 4e-6.
"""
import numpy as np
import pytest

import f64decoder as F
from qtts import synth

pytestmark = pytest.mark.gpu
TOL = 6.7e-5


@pytest.mark.parametrize("hidden,heads,inter,latent,frames", [
    (64, 1, 96, 64, (1, 15, 16, 17, 63, 64, 65, 300)),
    (512, 3, 160, 128, (2, 71, 72, 73, 129)),
    (576, 2, 1088, 320, (1, 3, 80, 257)),
])
def test_tf_rows(ctx_factory, hidden, heads, inter, latent, frames):
    d = synth.make_decoder(seed=67, latent=latent, hidden=hidden, n_heads=heads, head_dim=64, inter=inter, n_tf_layers=2,
                           codebook_size=64, codebook_dim=32, vq_dim=32, vocos=(96, 96), rates=(2,), dilations=(1,),
                           rope_max_pos=1024)
    ctx = ctx_factory(64)
    ctx.upload_decoder(d)
    assert ctx.debug_query("decoder_rows") == 3
    rng = np.random.Generator(np.random.PCG64(hidden))
    for T in frames:
        print(f"hidden {hidden} frames {T}", flush=True)
        codes = rng.integers(0, 64, (16, T)).astype(np.uint32)
        ref = F.decode(d, codes)
        got = ctx.decode_to_audio(codes)
        assert got.shape == ref.shape
        assert ctx.debug_query("decode_repeated") == 0
        err = np.abs(got.astype(np.float64) - ref).max() / np.abs(ref).max()
        assert err <= TOL, f"{T} frames: {err:.3g} of the largest sample"
