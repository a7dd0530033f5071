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


@pytest.mark.parametrize("n_cols", [1, 65535, 65536, 100003, 1179520])
@pytest.mark.parametrize("lanes", [1, 2, 4])
def test_layout_of_products_that_are_handed_bits(n_cols, lanes):
    """Every stored element is found again in the packed indices, everything else is the column past
    the end with the value -0; rows without elements and a short last slice included."""
    import scipy.sparse

    from nengo_ocl_amd import hipra_spmv as h

    rng = np.random.RandomState(n_cols)
    dense_rows = [np.unique(rng.randint(n_cols, size=k)) for k in rng.randint(0, 40, size=130)]
    dense_rows[0], dense_rows[129] = np.arange(0), np.array([n_cols - 1])
    mats = []
    for rows in (dense_rows, dense_rows[::-1][:70]):
        r = np.repeat(np.arange(len(rows)), [len(c) for c in rows])
        mats.append(h.HostSparseMatrix(scipy.sparse.csr_matrix(
            (1.0 + np.arange(len(r)), (r, np.concatenate(rows).astype(int))), shape=(len(rows), n_cols))))
    slice_rows, row_len, cols, vals = h.sell_layout(mats)
    starts, widths, packed, values, bits = h.bits_layout(slice_rows, row_len, cols, vals, n_cols, lanes)
    assert bits == (16 if n_cols < 65536 else 24) and not np.any(widths % (4 * lanes))
    if bits == 16:
        index = packed.view(np.uint16).astype(int)
    else:
        raw = np.ascontiguousarray(packed).view(np.uint8).reshape(-1, 3).astype(int)
        index = raw[:, 0] + 256 * raw[:, 1] + 65536 * raw[:, 2]
    assert len(index) == len(values) == int(np.sum(widths)) * 64
    used = np.zeros(len(values), dtype=bool)
    for (item, start, _, len_start, n_rows, row0), at in zip(slice_rows, starts):
        for r in range(n_rows):
            k = np.arange(row_len[len_start + r])
            new, old = h.sell_index(at, r, k), h.sell_index(start, r, k)
            used[new] = True
            assert np.array_equal(index[new], cols[old]) and np.array_equal(values[new], vals[old])
    assert np.all(index[~used] == n_cols) and np.all(np.signbit(values[~used])) and not np.any(values[~used])
