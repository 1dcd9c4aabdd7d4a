"""The fused kernels' loss tail over scenes of more than one chunk of 256 blocks:
its losses are the fixed-order mode's bits (both add the tiles' partials four to
a block, then blocks lane, lane + 64, ... per lane, then the lanes)."""

import numpy as np
import pytest

from diffrast import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from diffrast import _lib

    c = _lib.Context()
    yield c
    c.close()


# 256, 272, 512, 561 and 1071 blocks a scene
@pytest.mark.parametrize("H,W", [(256, 256), (257, 250), (512, 248), (513, 260), (1000, 270)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("B", [1, 2])
def test_tail_chunks(ctx, B, H, W):
    T, sigma = 24, 0.004
    params = synth.batch("random", B, T, 2200)
    bgs = synth.uniforms(2207, B * 3).reshape(B, 3).astype(np.float32)
    targets = np.stack([synth.blob_target(2200 + b, H, W) for b in range(B)])
    print(f"tail chunks B={B} {H}x{W}", flush=True)
    tail = ctx.fused_loss_backward(params, targets, sigma, bgs)[0]
    fixed = ctx.fused_loss_backward(params, targets, sigma, bgs, deterministic=True)[0]
    assert np.array_equal(tail, fixed)


# 1, 2, 16, 63, 64, 65, 128, 130 and 357 blocks a scene: one, two and four loads a lane, the last lanes without
@pytest.mark.parametrize("H,W", [(9, 16), (17, 5), (64, 64), (112, 131), (128, 128), (80, 200), (128, 256), (160, 208),
                                 (336, 272)], ids=lambda v: str(v))
@pytest.mark.parametrize("B", [1, 9])
def test_tail_of_small_scenes(ctx, B, H, W):
    T, sigma = 8, 0.01
    params = synth.batch("random", B, T, 2300)
    bgs = synth.uniforms(2307, B * 3).reshape(B, 3).astype(np.float32)
    targets = np.stack([synth.blob_target(2300 + b, H, W) for b in range(B)])
    print(f"tail of small scenes B={B} {H}x{W}", flush=True)
    tail = ctx.fused_loss_backward(params, targets, sigma, bgs)[0]
    fixed = ctx.fused_loss_backward(params, targets, sigma, bgs, deterministic=True)[0]
    assert np.array_equal(tail, fixed)
