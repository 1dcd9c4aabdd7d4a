"""The tile rows' lists (RowArgs), which the one-wave fused kernel's and the renders'
box tests read instead of every triangle's record: at images whose last tile row
and column are partial, triangles that end on tile edges, empty rows, NaN alpha
(drawn by a render, culled by the gradient paths) and more than one pass of 64
triangles a row, against the oracle.
"""

import numpy as np
import pytest

from bars import assert_grads, check_image, check_losses
from diffrast import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from diffrast import _lib

    c = _lib.Context()
    yield c
    c.close()


def aligned(params, H, W):
    """Every third triangle's vertices on 8-pixel lines, some of the others off the image."""
    p = params.copy()
    v = p[:, ::3, :6]
    v[..., 0::2] = np.round(v[..., 0::2] * W / 8) * 8 / W
    v[..., 1::2] = np.round(v[..., 1::2] * H / 8) * 8 / H
    p[:, ::3, :6] = v
    p[:, 1::11, :6] += np.float32(0.7)
    p[:, 2::11, :6] -= np.float32(0.7)
    return p.astype(np.float32)


# (B, H, W, T, sigma, kind): renders take rows from 128 triangles, gradients from
# 64 outside the segmented kernel (more than 2048 tiles for one scene, 6144 in a batch)
@pytest.mark.parametrize("B,H,W,T,sigma,kind", [
    (1, 393, 377, 64, 0.004, "random"),
    (1, 385, 400, 129, 0.001, "small"),
    (1, 400, 391, 300, 0.002, "random"),
    (2, 449, 460, 200, 0.0005, "small"),
    (1, 9, 4099, 140, 0.002, "small"),
    (1, 2500, 71, 140, 0.001, "small"),
], ids=lambda v: str(v))
def test_rows_match_oracle(ctx, orc, B, H, W, T, sigma, kind):
    params = aligned(synth.batch(kind, B, T, 3100), H, W)
    bgs = synth.uniforms(3107, B * 3).reshape(B, 3).astype(np.float32)
    targets = np.stack([synth.blob_target(3100 + b, H, W) for b in range(B)])
    print(f"row lists B={B} {H}x{W} T={T} {kind}", flush=True)
    img = orc.render_batch(params, H, W, sigma, bgs)
    check_image(ctx.render(params, H, W, sigma, bgs), img)
    gl, gg, gimg = ctx.fused_loss_backward(params, targets, sigma, bgs, want_images=True)
    check_image(gimg, img)
    cl, cg = orc.loss_backward_batch(params, targets, sigma, bgs)
    check_losses(gl, cl)
    assert_grads(gg, cg)


def test_nan_alpha_and_empty_rows(ctx, orc):
    # all triangles in a corner (most rows empty), some with a NaN alpha
    H, W, T, sigma = 400, 420, 150, 0.002
    params = synth.batch("small", 1, T, 3200)
    params[..., :6] = params[..., :6] * np.float32(0.2)
    params[:, ::13, 9] = np.nan
    bg = np.zeros((1, 3), np.float32)
    print("row lists with NaN alpha", flush=True)
    got, want = ctx.render(params, H, W, sigma, bg), orc.render_batch(params, H, W, sigma, bg)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    check_image(np.nan_to_num(got), np.nan_to_num(want))
    target = synth.blob_target(3200, H, W)[None]
    gl, gg = ctx.fused_loss_backward(params, target, sigma, bg)
    cl, cg = orc.loss_backward_batch(params, target, sigma, bg)
    check_losses(gl, cl)
    assert_grads(gg, cg)
