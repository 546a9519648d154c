"""The average over a whole image at the sizes where its kernel can go wrong: windows around the numbers of taps it keeps
under way, channel counts that fill no wave, one image and many.  The taps are added in the reference's order
(dabnn/layers/AvePool.cpp:84-123), so the result is the oracle's bit for bit."""
import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c", [
    (1, 1, 17, 1), (3, 4, 4, 64), (9, 4, 5, 3), (2, 31, 1, 64), (5, 4, 8, 66), (17, 3, 11, 5), (9, 7, 7, 512), (300, 7, 7, 20),
    (4, 5, 10, 63), (2, 7, 9, 65), (11, 8, 8, 256), (3, 5, 13, 7), (2, 9, 11, 100), (33, 16, 16, 256), (1, 56, 56, 64), (1, 1, 129, 4),
])
def test_average_over_the_whole_image(n, h, w, c):
    import dabnn_amd as dab
    x = np.random.default_rng(h * 100 + w).standard_normal((n, h, w, c)).astype(np.float32)
    x[-1, 0, 0, 0] = np.inf
    got = dab.ave_pool(torch.from_numpy(x).cuda(), h, w, 0, 0, 3, 2).cpu().numpy()
    sample = sorted({0, n // 2, n - 1})
    np.testing.assert_array_equal(got[sample], np.stack([orc.ave_pool(x[i], h, w, 0, 0, 3, 2) for i in sample]))
