"""drh_encode_srgb against the oracle where its table of runs could go wrong: the
first and last float of every run (the same exponent and first seven mantissa
bits), the floats around every threshold, values outside [0, 1], infinities and
every kind of NaN; and at counts and alignments around its four values per load.
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


def test_run_edges_and_specials(ctx, orc):
    runs = np.arange(0x3800, 0x3F90, dtype=np.uint32) << 16
    bits = np.concatenate([runs, runs + 1, runs + 0xFFFF, runs + 0x8000])
    special = np.array([0, 0x80000000, 0x80000001, 1, 0x00800000, 0x7F800000, 0xFF800000, 0x7FC00000, 0xFFC00000,
                        0x7F800001, 0xFF800001, 0x7FFFFFFF, 0x7F7FFFFF, 0xFF7FFFFF, 0xBF800000], np.uint32)
    # the floats around each byte's first value, from the oracle by bisection over the bits
    lo, hi = np.zeros(255, np.uint32), np.full(255, 0x3F800000, np.uint32)
    k = np.arange(1, 256)
    for _ in range(31):
        mid = lo + (hi - lo) // 2
        up = orc.encode_srgb(mid.view(np.float32)).astype(int) >= k
        hi, lo = np.where(up, mid, hi).astype(np.uint32), np.where(up, lo, mid).astype(np.uint32)
    near = np.concatenate([hi - 2, hi - 1, hi, hi + 1])
    values = np.concatenate([bits, special, near]).view(np.float32)
    assert np.array_equal(ctx.encode_srgb(values), orc.encode_srgb(values))


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 4097, 2048 * 256 * 4 + 7])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_counts_and_alignment(orc, n, shift):
    import torch

    from diffrast import _lib

    ctx = _lib.Context()
    x = torch.rand(n + 4, generator=torch.Generator().manual_seed(n)).mul_(1.2).sub_(0.1)
    d = x.cuda()
    out = torch.full((n + 8,), 77, dtype=torch.uint8, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    ctx.encode_srgb_ptr(d.data_ptr() + 4 * shift, n, out.data_ptr() + shift, s)
    got = out.cpu().numpy()
    assert np.array_equal(got[shift:shift + n], orc.encode_srgb(x.numpy()[shift:shift + n]))
    assert np.all(got[:shift] == 77) and np.all(got[shift + n:] == 77)
    ctx.close()
