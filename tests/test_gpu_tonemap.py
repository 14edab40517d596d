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
