"""Kernels whose decomposition depends on the size of a launch, at the sizes where that
decomposition has edges, against the CPU oracle bit for bit (every one of them keeps the
reference's order of summation, so the tolerance is zero)."""

import numpy as np
import pytest

from helpers import RA, to_dev

pytestmark = pytest.mark.gpu


# image (rows, columns, channels), filters, kernel, strides, padding: 64 to 800 chain links (16 read
# at a time), filters around the 16 of a wave and in whole quads or not, pixels around its 4
WAVE_CONV = [
    ((9, 4, 16), 33, (2, 2), (3, 1), (1, 0)),     # 64 links
    ((4, 4, 65), 1, (1, 1), (1, 1), "valid"),     # 65 links, one filter
    ((5, 5, 3), 3, (3, 11), (2, 1), "same"),      # 99 links, window wider than the image
    ((6, 7, 10), 16, (2, 4), (1, 1), "valid"),    # 80 links, 20 pixels
    ((12, 11, 13), 40, (3, 3), (2, 2), "same"),   # 117 links
    ((1, 1, 800), 20, (1, 1), (1, 1), "valid"),   # one pixel, as many links as fit
    ((2, 2, 801), 4, (1, 1), (1, 1), "valid"),    # one more: the tiles
    ((7, 7, 7), 17, (3, 3), (1, 1), "valid"),     # 63 links: the tiles
]


@pytest.mark.parametrize("case", WAVE_CONV)
def test_convolution_in_single_wave_groups(queue, rng, case):
    from nengo_ocl_amd import hipra_nonlinearities as nl
    from oracle import oracle as orc

    (nxi, nxj, nc), nf, (si, sj), (sti, stj), padding = case
    pi, pj = {"valid": (0, 0), "same": ((si - 1) // 2, (sj - 1) // 2)}.get(padding, padding)
    nyi, nyj = (nxi + 2 * pi - si) // sti + 1, (nxj + 2 * pj - sj) // stj + 1
    data = RA([rng.normal(size=5), rng.normal(size=nxi * nxj * nc),
               rng.normal(size=si * sj * nc * nf), rng.normal(size=nyi * nyj * nf),
               rng.normal(size=3)])
    dev = to_dev(queue, data)
    for mod, q, d in ((nl, queue, dev), (orc, None, data)):
        mod.plan_conv2d(q, d[[1]], d[[3]], d[[2]], (nxi, nxj, nc), (nyi, nyj, nf), (si, sj),
                        padding=padding, strides=(sti, stj), channels_last=True)()
    assert np.array_equal(dev.buf, data.buf)
