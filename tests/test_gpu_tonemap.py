"""The display pass against the oracle, bit for bit: ordinary pixels take the
short x^(1/2.2), a pixel with a zero, negative, infinite or NaN channel the
general one."""
import numpy as np
import pytest

import yune_amd as Y
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

ODD = np.float32([0.0, -0.0, -1.5, np.inf, -np.inf, np.nan, 1e-42, 1.4e-45, 3.4e38, 1.0, 1e-30])


@pytest.mark.parametrize("op", [Y.TONEMAP_REINHARD, Y.TONEMAP_HABLE])
@pytest.mark.parametrize("w,h", [(1, 1), (255, 1), (257, 3), (130, 97)])
def test_tonemap_matches_oracle(w, h, op):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(w * 7 + op)
    img = np.exp(rng.normal(-1.0, 3.0, (h, w, 4))).astype(np.float32)
    odd = rng.uniform(size=img.shape) < 0.02
    img[odd] = rng.choice(ODD, odd.sum())
    with Y.Context(max_paths=1 << 12) as c:
        a = torch.from_numpy(img).cuda()
        b = torch.empty_like(a)
        c.tonemap(b, a, w, h, op)
        got = b.cpu().numpy()
    want = O.tonemap(img, op)
    nan = np.isnan(want)
    assert np.array_equal(nan, np.isnan(got))
    assert np.array_equal(got[~nan].view(np.int32), want[~nan].view(np.int32))


@pytest.mark.parametrize("op", [Y.TONEMAP_REINHARD, Y.TONEMAP_HABLE])
def test_tonemap_over_the_floats_range(op):
    """Channels of every exponent (equal in a pixel, so that the others' size
    hides none of them), and around 1, where the logarithm's terms cancel."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(3 + op)
    wide = (rng.integers(1, 0x7F000000, 300_000).astype(np.uint32)).view(np.float32)
    near = np.float32(1) + np.arange(-50_000, 50_000, dtype=np.float32) * np.float32(2.0 ** -23)
    x = np.concatenate([wide, near, np.float32(2.0) ** np.arange(-126, 127, dtype=np.float32)])
    x = np.resize(x, (len(x) + 639) // 640 * 640)
    img = np.repeat(x[:, None], 4, 1).reshape(-1, 640, 4)
    img[1::3, :, 1] *= np.float32(0.5)
    img[2::3, :, 2] *= np.float32(1.7)
    with Y.Context(max_paths=1 << 12) as c:
        a = torch.from_numpy(img).cuda()
        b = torch.empty_like(a)
        torch.cuda.synchronize()
        c.tonemap(b, a, 640, len(img), op)
        got = b.cpu().numpy()
    want = O.tonemap(img, op)
    nan = np.isnan(want)
    assert np.array_equal(nan, np.isnan(got))
    assert np.array_equal(got[~nan].view(np.int32), want[~nan].view(np.int32))
    assert (want[~nan] > 0).mean() > 0.9 and nan.mean() < 0.3      # squares that overflow
