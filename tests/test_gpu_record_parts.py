"""The triangle records, which four lanes make together: every triangle count around the
16 records of a wave and the 128 of a workgroup beside an order, for one scene, for a
batch without a block order and for one with it, against the oracle. Equal records of the
three give equal images, bit for bit.
"""

import numpy as np
import pytest

from bars import check_image
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
