"""fused_seg_kernel over the sizes its rule takes (segment_waves): 8, 4 and 2
waves per tile, 16 to 1024 triangles, around the edges of its passes of 64
triangles, its block buffers and the entries a wave holds per pass.

Against the other kernels (DRH_NO_SEGMENTS=1): image and losses bit for bit, the
gradients to the order of their float sums; against the oracle at the usual bars.
"""

import numpy as np
import pytest

from bars import assert_grads, check_image, check_losses, grad_err
from diffrast import synth

pytestmark = pytest.mark.gpu

# (name, B, H, W, T, sigma, kind); tiles are 8x8, four to a 16x16 block
CASES = [
    # 8 waves: up to 768 tiles
    ("8w-T16", 1, 17, 23, 16, 0.004, "random"),
    ("8w-T64", 2, 40, 24, 64, 0.004, "uniform"),
    ("8w-T65", 1, 33, 48, 65, 0.01, "random"),
    ("8w-T161", 1, 61, 47, 161, 0.002, "random"),
    ("8w-T512", 1, 40, 40, 512, 0.01, "random"),
    ("8w-T513", 1, 24, 56, 513, 0.003, "small"),
    ("8w-T1024-long-lists", 1, 24, 24, 1024, 0.003, "uniform"),  # over 64 entries a wave
    # 4 waves: 768 to 2048 tiles, to 2560 in a batch, past 512 triangles below 6144
    ("4w-T17", 1, 232, 225, 17, 0.004, "random"),
    ("4w-T257", 3, 150, 155, 257, 0.004, "random"),
    ("4w-T600", 1, 230, 226, 600, 0.0015, "small"),
    ("4w-batch-T700", 12, 120, 130, 700, 0.003, "small"),
    # 2 waves: a batch of 2560 to 6143 tiles, from 48 triangles
    ("2w-T48", 11, 120, 130, 48, 0.004, "uniform"),
    ("2w-T66", 11, 120, 130, 66, 0.0015, "uniform"),
    ("2w-T200-long-lists", 11, 120, 130, 200, 0.002, "uniform"),
    ("2w-T512", 10, 121, 131, 512, 0.004, "random"),
    # just past the rule: the other kernels either way
    ("T1025", 1, 24, 24, 1025, 0.003, "small"),
    ("batch-T47", 11, 120, 130, 47, 0.004, "uniform"),
    ("batch-T16", 9, 128, 128, 16, 0.004, "random"),
]


@pytest.fixture(scope="module")
def ctx():
    from diffrast import _lib

    c = _lib.Context()
    yield c
    c.close()


def inputs(B, H, W, T, sigma, kind, seed=2100):
    params = synth.batch(kind, B, T, seed)
    params[:, ::7, 9] = 1.0  # exact zero factors where such a triangle covers a pixel
    bgs = synth.uniforms(seed + 7, B * 3).reshape(B, 3).astype(np.float32)
    targets = np.stack([synth.blob_target(seed + b, H, W) for b in range(B)])
    return params, bgs, targets


@pytest.mark.parametrize("name,B,H,W,T,sigma,kind", CASES, ids=[c[0] for c in CASES])
def test_sizes_match_other_kernels(ctx, orc, name, B, H, W, T, sigma, kind, monkeypatch):
    params, bgs, targets = inputs(B, H, W, T, sigma, kind)
    print(f"segment sizes {name}", flush=True)
    gin = ((synth.uniforms(9, B * H * W * 3) - 0.5) * 1e-3).reshape(B, H, W, 3).astype(np.float32)

    def all_modes():
        gl, gg, gimg = ctx.fused_loss_backward(params, targets, sigma, bgs, want_images=True)
        dl, dg = ctx.fused_loss_backward(params, targets, sigma, bgs, deterministic=True)
        el, eg = ctx.fused_loss_backward(params, targets, sigma, bgs, exact=True)
        return gl, gg, gimg, dl, dg, el, eg, ctx.backward_from_grad(params, gin, sigma, bgs)

    gl, gg, gimg, dl, dg, el, eg, fg = all_modes()
    again = ctx.fused_loss_backward(params, targets, sigma, bgs, deterministic=True)
    assert np.array_equal(again[0], dl) and np.array_equal(again[1], dg)
    monkeypatch.setenv("DRH_NO_SEGMENTS", "1")
    ol, og, oimg, odl, odg, oel, oeg, ofg = all_modes()
    assert np.array_equal(gimg, oimg) and np.array_equal(gl, ol)
    assert np.array_equal(dl, odl) and np.array_equal(dl, gl) and np.array_equal(el, oel)
    # float sums in another order: 2^-24 relative per addition, a few hundred of them
    for a, b in ((gg, og), (dg, odg), (eg, oeg), (fg, ofg)):
        assert grad_err(a, b) <= 2e-6
    cl, cg = orc.loss_backward_batch(params, targets, sigma, bgs)
    check_image(gimg, orc.render_batch(params, H, W, sigma, bgs), label=name)
    check_losses(gl, cl, label=name)
    assert_grads(gg, cg, label=name)
    assert_grads(dg, cg, label=f"{name} fixed order")

