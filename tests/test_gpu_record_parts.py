"""The triangle records, which four lanes make together: every triangle count around the
16 records of a wave and the 128 of a workgroup beside an order, for one scene, for a
batch without a block order and for one with it, against the oracle. Equal records of the
three give equal images, bit for bit.
"""

import numpy as np
import pytest

from bars import assert_grads, check_image, check_losses
from diffrast import synth

pytestmark = pytest.mark.gpu

SIGMA = 0.003
H, W = 72, 88  # 30 blocks: 16 scenes have more than the device has CUs


@pytest.fixture(scope="module")
def ctx():
    from diffrast import _lib

    c = _lib.Context()
    yield c
    c.close()


@pytest.mark.parametrize("T", [1, 3, 15, 16, 17, 33, 127, 128, 129, 257])
def test_record_counts(ctx, orc, T):
    print(f"record parts T={T}", flush=True)
    params = synth.batch("random", 2, T, 4100)
    params[:, 1::5, 4:6] = params[:, 1::5, 2:4]  # an edge of no length
    params[1, ::7, 9] = 0.0
    bgs = synth.uniforms(4107, 6).reshape(2, 3).astype(np.float32)
    two = ctx.render(params, H, W, SIGMA, bgs)
    check_image(two, orc.render_batch(params, H, W, SIGMA, bgs))
    many = ctx.render(np.tile(params, (8, 1, 1)), H, W, SIGMA, np.tile(bgs, (8, 1)))
    for i in range(16):
        assert np.array_equal(many[i], two[i % 2])
    for b in range(2):
        assert np.array_equal(ctx.render(params[b:b + 1], H, W, SIGMA, bgs[b:b + 1])[0], two[b])


@pytest.mark.parametrize("T", [1537, 1700, 3000])
def test_records_in_two_strides(ctx, orc, T):
    # 16 scenes of 8 tile rows: 8 + T / 64 setup workgroups each, past 512 in all from 1537
    # triangles (64 a workgroup); a scene alone takes its records in one stride
    H, W = 64, 60
    print(f"record strides T={T}", flush=True)
    params = synth.batch("small", 2, T, 4200)
    bgs = synth.uniforms(4207, 6).reshape(2, 3).astype(np.float32)
    targets = np.stack([synth.blob_target(4200 + b, H, W) for b in range(2)])
    many = [np.tile(x, (8,) + (1,) * (x.ndim - 1)) for x in (params, targets, bgs)]
    img = ctx.render(many[0], H, W, SIGMA, many[2])
    losses, grads = ctx.fused_loss_backward(many[0], many[1], SIGMA, many[2])
    want = orc.loss_backward_batch(params, targets, SIGMA, bgs)
    for b in range(2):
        one = ctx.render(params[b:b + 1], H, W, SIGMA, bgs[b:b + 1])[0]
        check_image(one[None], orc.render_batch(params[b:b + 1], H, W, SIGMA, bgs[b:b + 1]))
        for i in range(b, 16, 2):
            assert np.array_equal(img[i], one)
            check_losses(losses[i:i + 1], want[0][b:b + 1])
            assert_grads(grads[i:i + 1], want[1][b:b + 1])
