"""Which kernel a launch takes, by its sizes: rules that can be followed without a device."""

import numpy as np
import pytest


def conv_threads(shape_in, filters, kernel, strides=(1, 1), channels_last=True, conv=True):
    """Threads per group for an unpadded convolution, after a look at the number of groups."""
    from nengo_ocl_amd import _lib
    from nengo_ocl_amd import hipra_nonlinearities as nl

    (nxi, nxj, nc), (si, sj), (sti, stj) = shape_in, kernel, strides
    nyi, nyj = (nxi - si) // sti + 1, (nxj - sj) // stj + 1
    tiles = nl.conv2d_tiles((nyi, nyj, filters), kernel, strides, nc, channels_last)
    geom = np.array([nxi, nxj, nc, nyi, nyj, filters, si, sj, sti, stj, 0, 0, 0, 0, 0,
                     int(channels_last), int(not conv), *tiles], dtype=np.int32)
    n_tiles = -(-nyi // tiles[0]) * -(-nyj // tiles[1]) * -(-filters // tiles[2])
    n_waves = -(-nyi * nyj // 4) * -(-filters // 16)
    groups, threads = nl.conv2d_groups(_lib.lib(), geom)
    assert groups == {256: n_tiles, 64: n_waves}[threads]
    return threads


@pytest.mark.parametrize("channels_last,conv,expected", [(True, True, 64), (False, True, 256),
                                                         (True, False, 256)])
def test_launch_size_of_a_convolution_is_that_of_its_kernel(channels_last, conv, expected):
    assert conv_threads((26, 26, 32), 64, (3, 3), (2, 2), channels_last, conv) == expected
    assert conv_threads((26, 26, 3), 64, (3, 3), (2, 2), channels_last, conv) == 256  # 27 links


# image, filters, kernel, strides; what the other kernel would cost (measured) stands beside the rule
@pytest.mark.parametrize("shape_in,filters,kernel,strides,expected", [
    ((46, 46, 40), 80, (3, 3), (2, 2), 64), ((10, 10, 8), 16, (3, 3), (2, 2), 64),
    ((28, 28, 32), 256, (3, 3), (1, 1), 64), ((64, 64, 32), 2, (3, 3), (1, 1), 64),
    ((128, 128, 32), 2, (3, 3), (1, 1), 256), ((512, 512, 88), 1, (3, 3), (1, 1), 256),
    ((256, 256, 8), 4, (3, 3), (1, 1), 256), ((28, 28, 3), 16, (5, 5), (2, 2), 256),
    ((200, 200, 16), 64, (7, 7), (2, 2), 256), ((64, 64, 88), 64, (3, 3), (1, 1), 256),
    ((64, 64, 200), 256, (1, 1), (1, 1), 64), ((256, 256, 400), 2, (1, 1), (1, 1), 256),
    ((20, 20, 801), 2, (1, 1), (1, 1), 256)])
def test_convolutions_take_single_wave_groups_where_these_are_resident(shape_in, filters, kernel,
                                                                       strides, expected):
    assert conv_threads(shape_in, filters, kernel, strides) == expected
