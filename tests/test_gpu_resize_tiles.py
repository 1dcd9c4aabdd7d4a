"""drh_resize_lanczos3's one-kernel form (resize_tile) and the two kernels that it
falls back to, byte for byte against the oracle: rows of whole and of partial
words, one to four channels, output widths around its chunks of columns, windows
up to and past its LDS, more rows than a grid has.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from diffrast import _lib

    c = _lib.Context()
    yield c
    c.close()


@pytest.mark.parametrize("shape,size", [
    ((600, 800, 3), (176, 132)), ((601, 797, 3), (150, 113)), ((300, 333, 1), (31, 29)), ((200, 222, 2), (65, 33)),
    ((150, 151, 4), (64, 64)), ((64, 64, 3), (513, 40)), ((40, 50, 3), (1025, 700)), ((37, 41, 3), (1, 1)),
    ((3, 1700, 3), (1, 2)), ((4, 3000, 4), (2, 3)), ((2, 40000, 3), (2, 2)), ((3, 40001, 1), (1, 5)),
    ((90000, 4, 1), (2, 70000)),
], ids=lambda v: "x".join(map(str, v)))
def test_resize_tiles(ctx, orc, shape, size):
    img = np.random.default_rng(shape[0] + 7 * size[0]).integers(0, 256, shape, dtype=np.uint8)
    print(f"resize tiles {shape} -> {size}", flush=True)
    assert np.array_equal(ctx.resize_lanczos3(img, *size), orc.resize_lanczos3(img, *size))


@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_unaligned_device_image(orc, shift):
    import torch

    from diffrast import _lib

    ctx = _lib.Context()
    H, W, C, nh, nw = 120, 164, 3, 33, 40
    img = np.random.default_rng(shift).integers(0, 256, (H, W, C), dtype=np.uint8)
    buf = torch.zeros(H * W * C + 8, dtype=torch.uint8)
    buf[shift:shift + H * W * C] = torch.from_numpy(img.reshape(-1))
    buf = buf.cuda()
    out = torch.full((nh * nw * C + 8,), 9, dtype=torch.uint8, device="cuda")
    ctx.resize_lanczos3_ptr(buf.data_ptr() + shift, H, W, C, out.data_ptr() + shift, nh, nw,
                            torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.array_equal(got[shift:shift + nh * nw * C].reshape(nh, nw, C), orc.resize_lanczos3(img, nw, nh))
    assert np.all(got[:shift] == 9) and np.all(got[shift + nh * nw * C:] == 9)
    ctx.close()
