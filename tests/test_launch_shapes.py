"""Kernels whose decomposition depends on the size of a launch, at the sizes where that
decomposition has edges, against the CPU oracle bit for bit (every one of them keeps the
reference's order of summation, so the tolerance is zero)."""

import numpy as np
import pytest

from helpers import RA, clone, run_plans, to_dev

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


@pytest.mark.parametrize("rows,cols,per_row", [
    (1, 1, 1), (17, 64, 12), (64 * 63 + 49, 65, 3), (64 * 256 + 1, 1000, 12), (300, 32768, 64),
    (300, 32769, 130), (130, 900, 16), (97, 5000, 300)])
def test_sparse_product_of_spikes_spread_over_the_device(queue, rng, monkeypatch, rows, cols,
                                                         per_row):
    """Fewer and more quarters of slices than waves of the device; rows of one quad to several
    batches of them; the bits of X formed by the groups themselves (up to 32,768 elements) and
    by a launch of their own; sums that are negative zeros."""
    import scipy.sparse as sp

    from nengo_ocl_amd import hipra_spmv
    from oracle import oracle as orc

    monkeypatch.setattr(hipra_spmv, "SKIP_MIN_WIDTH", 0)  # short rows too
    mat = sp.random(rows, cols, density=min(1.0, per_row / cols), random_state=3, format="csr",
                    dtype=np.float32)
    X = RA([np.zeros(3), np.where(rng.uniform(size=cols) < 0.2, rng.normal(size=cols), 0.0)])
    Y = RA([np.where(np.arange(rows) % 3 == 0, -0.0, rng.normal(size=rows))])
    dX, dY, Yo = to_dev(queue, X), to_dev(queue, Y), clone(Y)
    prog = hipra_spmv.plan_sparse_dot_inc(queue, [mat], dX[[1]], dY, inc=True, x_mostly_zero=True)
    assert prog.plans[0].skips_zero_x
    oplan = orc.plan_sparse_dot_inc(None, [mat], X[[1]], Yo, inc=True).plans[0]
    # many values, one value (as spikes of one amplitude have), none, one negative value
    for x in (X[1], 1000.0 * (X[1] != 0), 0.0 * X[1] + 0.0, -2.5 * (X[1] > 0) + 0.0):
        X[1] = x
        dX[1] = x
        prog.plans[0]()
        oplan()
        assert np.array_equal(dY.buf.view(np.uint32), Yo.buf.view(np.uint32))


@pytest.mark.parametrize("cols", [32768, 32769])
def test_sparse_product_without_ranges(queue, rng, cols):
    """`nhip_spmv_sell_skip` writes no more than the one bit per element that its workspace holds,
    and what it gives is the ordinary product."""
    import scipy.sparse as sp

    from nengo_ocl_amd import hipra_spmv
    from nengo_ocl_amd.hipraggedarray import to_device

    rows = 300
    mat = sp.random(rows, cols, density=40 / cols, random_state=3, format="csr", dtype=np.float32)
    X = RA([np.where(rng.uniform(size=cols) < 0.1, 1000.0, 0.0)])
    Y = RA([rng.normal(size=rows)])
    dX, dY, dY2 = to_dev(queue, X), to_dev(queue, Y), to_dev(queue, Y)
    plan = hipra_spmv.plan_sparse_dot_inc(queue, [mat], dX, dY, inc=True).plans[0]
    plan()
    words = -(-cols // 128) * 4
    mask = to_device(queue, np.full(words + 256, 77, dtype=np.int32))
    args = plan.args[:6] + (dY2.ptr, int(dX.starts[0]), cols, mask.ptr)
    assert queue.lib.nhip_spmv_sell_skip(queue.handle, *args) == 0
    assert np.array_equal(dY.buf.view(np.uint32), dY2.buf.view(np.uint32))
    assert (mask.get()[words:] == 77).all()


@pytest.mark.parametrize("padding", ["values", "values and columns"])
@pytest.mark.parametrize("rows,cols,longest", [
    (64 * 40 + 21, 900, 14), (64 * 40 + 21, 40000, 14), (64 * 40 + 21, 900, 150),
    (64 * 40 + 21, 40000, 150),
    (64 * 1830 + 1, 900, 14), (64 * 3300 + 7, 40000, 29)])  # (whole slices)
def test_sparse_product_ignores_what_is_stored_past_a_rows_end(queue, rng, rows, cols, longest,
                                                               padding):
    """Rows are padded to the longest of their slice: no entry point may look at what the padding
    holds, neither as a factor (infinities, NaN, negative numbers, with sums of -0 among the results)
    nor as an index."""
    import scipy.sparse as sp

    from nengo_ocl_amd import hipra_spmv
    from nengo_ocl_amd.hipraggedarray import to_device
    from oracle import oracle as orc

    lens = rng.randint(0, longest + 1, size=rows)
    lens[::64] = longest
    indptr = np.concatenate([[0], np.cumsum(lens)])
    mat = sp.csr_matrix((rng.normal(size=indptr[-1]).astype(np.float32),
                         rng.randint(cols, size=indptr[-1]), indptr), shape=(rows, cols))
    mat.sum_duplicates()
    host = hipra_spmv.HostSparseMatrix(mat)
    slice_rows, row_len, cidx, vals = hipra_spmv.sell_layout([host])
    padded = np.ones(vals.size, dtype=bool)
    for _, start, width, len_start, n_rows, _ in slice_rows:
        at = hipra_spmv.sell_index(start, np.arange(64)[:, None], np.arange(width))
        padded[at] = np.arange(width) >= row_len[len_start:len_start + 64][:, None]
    vals[padded] = rng.choice([np.nan, np.inf, -np.inf, -3.0], size=padded.sum())
    if padding != "values":
        cidx[padded] = 2 ** 31 - 1
    X = RA([np.where(rng.uniform(size=cols) < 0.2, rng.normal(size=cols), 0.0)])
    Y = RA([np.where(np.arange(rows) % 2 == 0, -0.0, rng.normal(size=rows))])
    dX = to_dev(queue, X)
    table = np.zeros((len(slice_rows), 8), dtype=np.int32)
    for k, (_, start, width, len_start, n_rows, row0) in enumerate(slice_rows):
        table[k] = (start, width, len_start, n_rows, int(dX.starts[0]), row0, 1, -1)
    d = [to_device(queue, a) for a in (table, row_len, cidx, vals)]
    words = -(-cols // 128) * 4
    mask, ranges = (to_device(queue, np.zeros(words, dtype=np.int32)) for _ in range(2))
    head = (d[0].ptr, len(table), d[1].ptr, d[2].ptr, d[3].ptr, dX.ptr)
    none, span, lib = (None, None, None), (int(dX.starts[0]), cols), queue.lib
    calls = {"nhip_spmv_sell": (), "nhip_spmv_sell_skip": span + (mask.ptr,),
             "nhip_spmv_sell_spikes": none + span + (mask.ptr, ranges.ptr)}
    for x in (X[0], 1000.0 * (X[0] != 0)):  # many values, one value
        X[0] = x
        dX[0] = x
        Yo = clone(Y)
        orc.plan_sparse_dot_inc(None, [mat], X, Yo, inc=True).plans[0]()
        for name, rest in calls.items():
            dY = to_dev(queue, Y)
            assert getattr(lib, name)(queue.handle, *head, dY.ptr, *rest) == 0
            queue.finish()
            assert np.array_equal(dY.buf.view(np.uint32), Yo.buf.view(np.uint32)), name


# (on 256 compute units: from 0.8 slices per wave on, not just above one per wave, from 1.5 on; of short
# rows from 0.45 on)
@pytest.mark.parametrize("rows,cols,per_row", [
    (64 * 1821 + 5, 3000, 7), (64 * 3277 + 50, 40000, 40), (64 * 4096, 32768, 26),
    (64 * 4096 + 1, 70000, 26), (64 * 6144 + 63, 600, 28)])
def test_sparse_product_of_spikes_in_whole_slices(queue, rng, monkeypatch, rows, cols, per_row):
    """As many slices as waves, and more: with a filter behind the rows, X of many values and of one."""
    import scipy.sparse as sp

    from nengo_ocl_amd import hipra_nonlinearities as nl
    from nengo_ocl_amd import hipra_spmv
    from oracle import oracle as orc

    monkeypatch.setattr(hipra_spmv, "SKIP_MIN_WIDTH", 0)
    lens = rng.randint(0, per_row + 1, size=rows)
    lens[::64] = per_row
    indptr = np.concatenate([[0], np.cumsum(lens)])
    mat = sp.csr_matrix((rng.normal(size=indptr[-1]).astype(np.float32),
                         rng.randint(cols, size=indptr[-1]), indptr), shape=(rows, cols))
    mat.sum_duplicates()
    R = RA([np.where(rng.uniform(size=cols) < 0.2, rng.normal(size=cols), 0.0),
            np.where(np.arange(rows) % 3 == 0, -0.0, rng.normal(size=rows)), rng.normal(size=rows)])
    den, num = RA([np.array([[-0.8]])]), RA([np.array([[0.2]])])
    dev, host = to_dev(queue, R), clone(R)
    bufs = [RA([np.zeros((1, rows))]) for _ in range(2)]
    plans = []
    for ra, spmv, mod, q, up, kw in (
            (dev, hipra_spmv.plan_sparse_dot_inc, nl, queue, lambda a: to_dev(queue, a),
             dict(x_mostly_zero=True)),
            (host, orc.plan_sparse_dot_inc, orc, None, clone, {})):
        plans.append((spmv(q, [mat], ra[[0]], ra[[1]], inc=True, **kw).plans[0],
                      mod.plan_linearfilter(q, ra[[1]], ra[[2]], up(den), up(num), up(bufs[0]),
                                            up(bufs[1]))))
    (plan, lf), (oplan, olf) = plans
    assert plan.skips_zero_x
    fused, residual = hipra_spmv.fuse_linearfilter(plan, lf[0])
    assert [p.name for p in fused] == ["hip_spmv_filter"] and not residual
    for x in (R[0], 1000.0 * (R[0] != 0)):
        dev[0] = x
        host[0] = x
        run_plans(fused)
        oplan()
        run_plans(olf)
        assert np.array_equal(dev.buf.view(np.uint32), host.buf.view(np.uint32))


# short rows: enough of them in all, or the ordinary launch
@pytest.mark.parametrize("rows,cols,per_row,skips", [
    (150000, 150000, 12, True), (440000, 40000, 4, True), (430000, 40000, 4, False),
    (70000, 70000, 24, False), (3000, 3000, 28, True), (3000, 3000, 24, False)])
def test_sparse_product_of_spikes_with_short_rows(queue, rng, rows, cols, per_row, skips):
    import scipy.sparse as sp

    from nengo_ocl_amd import hipra_nonlinearities as nl
    from nengo_ocl_amd import hipra_spmv
    from oracle import oracle as orc

    columns = np.sort(rng.randint(cols - per_row, size=(rows, per_row)), axis=1) + np.arange(per_row)
    mat = sp.csr_matrix((rng.normal(size=columns.size).astype(np.float32), columns.ravel(),
                         np.arange(0, columns.size + 1, per_row)), shape=(rows, cols))
    R = RA([np.where(rng.uniform(size=cols) < 0.1, 1000.0, 0.0), rng.normal(size=rows),
            rng.normal(size=rows)])
    dev, host = to_dev(queue, R), clone(R)
    den, num, zero = RA([np.array([[-0.8]])]), RA([np.array([[0.2]])]), RA([np.zeros((1, rows))])
    plan = hipra_spmv.plan_sparse_dot_inc(queue, [mat], dev[[0]], dev[[1]], inc=True,
                                          x_mostly_zero=True).plans[0]
    assert plan.skips_zero_x == skips
    up = lambda a: to_dev(queue, a)
    lf = nl.plan_linearfilter(queue, dev[[1]], dev[[2]], up(den), up(num), up(zero), up(zero))
    fused, residual = hipra_spmv.fuse_linearfilter(plan, lf[0])
    assert not residual
    run_plans([plan] + fused)
    oplan = orc.plan_sparse_dot_inc(None, [mat], host[[0]], host[[1]], inc=True).plans[0]
    run_plans([oplan, oplan] + orc.plan_linearfilter(None, host[[1]], host[[2]], den, num, clone(zero),
                                                     clone(zero)))
    assert np.array_equal(dev.buf.view(np.uint32), host.buf.view(np.uint32))


@pytest.mark.parametrize("widths", [
    [512, 513, 639, 2047, 2048, 2049, 4095, 4096, 4097, 6145, 9216, 640, 8193],
    [512, 513, 514, 515, 639, 2047, 2048, 1920, 1921, 1999, 2000, 640, 2046],
    [160, 161, 162, 163, 255, 256, 257, 383, 384, 385, 511, 512, 200]],
    ids=["group per row", "wave per row", "short rows"])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_few_long_rows(queue, rng, beta, widths):
    """Widths around the 128-column tiles and around the columns of one pass of a wave (2,048)
    and of a group (8,192)."""
    from nengo_ocl_amd import hipra_gemv
    from oracle import oracle as orc

    heights = [33, 1, 2, 17, 10, 3, 5, 40, 1, 2, 10, 70, 1]
    A = RA([rng.normal(size=(m, n)) for m, n in zip(heights, widths)])
    X = RA([rng.normal(size=n) for n in widths])
    Y = RA([rng.normal(size=m) for m in heights])
    A_js = RA([[k] for k in range(len(widths))], dtype=np.int32)
    dA, dX, dY, Yo = to_dev(queue, A), to_dev(queue, X), to_dev(queue, Y), clone(Y)
    args = lambda a, x: (1.5, a, A_js, x, A_js, beta)
    prog = hipra_gemv.plan_block_gemv(queue, *args(dA, dX), dY, gamma=0.25)
    long_rows = [p for p in prog.plans if p.kernel_class[:2] in ((2, hipra_gemv.LONG_ROWS), (2, 256))]
    assert long_rows == prog.plans and len(long_rows) == 1
    run_plans(prog.plans)
    orc.plan_block_gemv(None, *args(A, X), Yo, gamma=0.25).plans[0]()
    assert np.array_equal(dY.buf.view(np.uint32), Yo.buf.view(np.uint32))


@pytest.mark.parametrize("heights,widths,lanes", [
    ([1, 700, 200, 60, 62], [512, 516, 2048, 2044, 2052], 128), ([400, 624, 1], [1000, 640, 513], 128),
    ([1024], [2056], 128)])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_long_rows_in_quads(queue, rng, heights, widths, lanes, beta):
    """Rows that fill the device and lie on 16-byte boundaries, in whole quads or not, around the tiles and
    the passes; sums that are or start at -0, and an infinity beside the last tile's end."""
    from nengo_ocl_amd import hipra_gemv
    from oracle import oracle as orc

    A = RA([rng.normal(size=(m, n)) for m, n in zip(heights, widths)], align=True)
    X = RA([rng.normal(size=n) for n in widths], align=True)
    Y = RA([-0.0 * np.ones(m) for m in heights], align=True)
    A[0][0, :] = -1e-45
    X[0][:] = 1e-3
    A[len(widths) - 1][-1, -1] = np.inf
    A_js = RA([[k] for k in range(len(widths))], dtype=np.int32)
    dA, dX, dY, Yo = to_dev(queue, A), to_dev(queue, X), to_dev(queue, Y), clone(Y)
    prog = hipra_gemv.plan_block_gemv(queue, 1.5, dA, A_js, dX, A_js, beta, dY)
    assert [p.kernel_class for p in prog.plans] == [(2, lanes, 1)]
    run_plans(prog.plans)
    orc.plan_block_gemv(None, 1.5, A, A_js, X, A_js, beta, Yo).plans[0]()
    assert np.array_equal(dY.buf.view(np.uint32), Yo.buf.view(np.uint32))


@pytest.mark.parametrize("pre,dims,lanes", [(1000, 200, 128), (5000, 2100, 256)],
                         ids=["wave per row", "group per row"])
def test_few_long_rows_with_epilogues(queue, pre, dims, lanes):
    """Encoders of many dimensions and decoders of many neurons: long rows whose launch also updates the
    neurons or steps the filters, and carries a sequence, bit for bit like the oracle's; class and
    tag tell them from large-item launches of the same name."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        rng = np.random.RandomState(5)
        net = mb.Network(seed=4, solver="surrogate")
        stim = net.Node(mb.WhiteSignal(period=0.5, high=8.0, seed=3), size_out=2)
        a = net.Ensemble(pre, 2, neuron_type=mb.LIFRate())
        net.Connection(stim, a, synapse=None)
        out = net.Node(None, size_in=3)
        net.Connection(a.neurons, out, synapse=mb.Lowpass(0.005),
                       transform=rng.normal(scale=1e-2 / pre, size=(3, pre)))
        wide = net.Ensemble(250, dims, radius=3.0)
        net.Connection(stim, wide, synapse=mb.Lowpass(0.01), transform=rng.normal(size=(dims, 2)))
        return net, [net.Probe(out), net.Probe(wide.neurons)]

    (net, probes), (net_o, probes_o) = make(), make()
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        rows = {p.name: p for p in gpu._plans if getattr(p, "kernel_class", ()) == (2, lanes, 1)}
        assert set(rows) == {"hipra_gemv.tile_lif", "hipra_gemv.tile_filter"}
        assert all("long-rows%d" % lanes in p.tag for p in rows.values())
        assert not any("long-rows" in p.tag for p in gpu._plans if p not in rows.values() and p.tag)
        assert any(getattr(p, "carried", None) is not None for p in rows.values())
        gpu.run_steps(60)
        cpu.run_steps(60)
        for p, q in zip(probes, probes_o):
            assert np.array_equal(gpu.data[p], cpu.data[q]) and np.any(gpu.data[p] != 0)
        assert np.array_equal(gpu.signal_buffer(), cpu.signal_buffer())


@pytest.mark.parametrize("rows,cols", [(1, 700), (503, 700), (1, 5000), (300, 5000)])
def test_few_long_rows_carry_a_sequence(queue, rng, rows, cols):
    """Two chains in groups of their own beside those of the rows, which have no epilogue."""
    from nengo_ocl_amd import hipra_gemv, hipra_sequence
    from nengo_ocl_amd import hipra_nonlinearities as nl
    from oracle import oracle as orc

    A, X, Y = RA([rng.normal(size=(rows, cols))]), RA([rng.normal(size=cols)]), RA([rng.normal(size=rows)])
    C = RA([rng.normal(size=50) for _ in range(4)])
    js = RA([[0]], dtype=np.int32)
    dA, dX, dY, dC, Yo = *(to_dev(queue, v) for v in (A, X, Y, C)), clone(Y)
    plan, = hipra_gemv.plan_block_gemv(queue, 1.5, dA, js, dX, js, 1.0, dY).plans
    copies = [nl.plan_copy(queue, dC[[k]], dC[[k + 2]], [1]) for k in range(2)]
    plan.reads_mem, plan.writes_mem = {"A", "X"}, {"Y"}
    for k, p in enumerate(copies):
        p.reads_mem, p.writes_mem = {k}, {k + 2}
    carrier, = hipra_sequence.carry_sequences([plan, hipra_sequence.plan_sequence(queue, copies)])
    assert carrier is plan and plan.kernel_class[0] == 2 and plan.carried is not None
    plan()
    orc.plan_block_gemv(None, 1.5, A, js, X, js, 1.0, Yo).plans[0]()
    assert np.array_equal(dY.buf.view(np.uint32), Yo.buf.view(np.uint32))
    for k in range(2):
        assert np.array_equal(dC[k + 2], np.float32(C[k]) + np.float32(C[k + 2]))


# rows, columns, elements between rows, of a buffer's start, and pre's stride: four elements of a row
# at a time or not, rows shorter and longer than a block of 1024, one element, blocks with a rest
LEARN_SHAPES = [(1, 1, 1, 0, 1), (3, 4, 4, 0, 1), (257, 4, 8, 4, 1), (5, 1028, 1028, 0, 1),
                (129, 100, 100, 0, 2), (129, 100, 104, 2, 1), (129, 100, 101, 0, 1),
                (41, 255, 255, 0, 1), (2, 2050, 2052, 0, 1)]


@pytest.mark.parametrize("inc", [False, True])
@pytest.mark.parametrize("rule", ["bcm", "oja", "voja"])
@pytest.mark.parametrize("shape", LEARN_SHAPES)
def test_learning_rule_in_quads_of_a_row(queue, rng, rule, inc, shape):
    """The change of a matrix, stored apart or added to the matrix it is formed from."""
    from nengo_ocl_amd import hipra_nonlinearities as nl
    from nengo_ocl_amd.hipraggedarray import HIPRaggedArray
    from nengo_ocl_amd.raggedarray import RaggedArray
    from oracle import oracle as orc

    m, n, stride, shift, pre_stride = shape
    sizes = [4 + m * stride, 4 + m * stride, 4 + n * pre_stride, m, m, 1, m]
    big = RA([rng.uniform(-2, 9, size=k) for k in sizes])
    dbig = to_dev(queue, big)
    s = big.starts
    at = dict(pre=(s[2] + shift, n, 1, pre_stride), post=(s[3], m, 1, 1), theta=(s[4], m, 1, 1),
              learn=(s[5], 1, 1, 1), scale=(s[6], m, 1, 1), mat=(s[0] + shift, m, n, stride),
              delta=(s[0 if inc else 1] + shift, m, n, stride))
    views = []
    for d in (False, True):
        one = lambda *v: [np.int32([x]) for x in v]
        views.append({k: HIPRaggedArray.from_buffer(queue, dbig.dev_buf, *one(*v, 1)) if d else
                      RaggedArray.from_buffer(big.buf, *one(*v, 1)) for k, v in at.items()})
    alpha, beta = np.float32([1e-3]), np.float32([1.5])
    for mod, q, v in ((orc, None, views[0]), (nl, queue, views[1])):
        if rule == "bcm":
            mod.plan_bcm(q, v["pre"], v["post"], v["theta"], v["delta"], alpha, inc=inc)()
        elif rule == "oja":
            mod.plan_oja(q, v["pre"], v["post"], v["mat"], v["delta"], alpha, beta, inc=inc)()
        else:
            mod.plan_voja(q, v["pre"], v["post"], v["mat"], v["delta"], v["learn"], v["scale"], alpha,
                          inc=inc)()
    assert np.array_equal(dbig.buf.view(np.uint32), big.buf.view(np.uint32))


@pytest.mark.parametrize("heights,cols,four_lanes", [
    ([8193], 1, True), ([2731, 8192], 3, True), ([65535], 1, True), ([9001, 40, 3], 2, True),
    ([8193], 5, False), ([65536], 1, False)])
def test_many_rows_of_few_columns(queue, rng, heights, cols, four_lanes):
    """Just above the small items' limit, and up to the rows that get a lane each."""
    from nengo_ocl_amd import hipra_gemv
    from oracle import oracle as orc

    A = RA([rng.normal(size=(m, cols)) for m in heights])
    X = RA([rng.normal(size=cols) for _ in heights])
    Y = RA([rng.normal(size=m) for m in heights])
    js = RA([[k] for k in range(len(heights))], dtype=np.int32)
    dA, dX, dY, Yo = to_dev(queue, A), to_dev(queue, X), to_dev(queue, Y), clone(Y)
    prog = hipra_gemv.plan_block_gemv(queue, 1.5, dA, js, dX, js, 1.0, dY, gamma=0.25)
    assert ([p.kernel_class[:3] for p in prog.plans] == [(2, 4, 1)]) == four_lanes
    run_plans(prog.plans)
    orc.plan_block_gemv(None, 1.5, A, js, X, js, 1.0, Yo, gamma=0.25).plans[0]()
    assert np.array_equal(dY.buf.view(np.uint32), Yo.buf.view(np.uint32))


# ensembles of as many neurons as make the tasks of every kind of neuron launch start at multiples of
# 32 rows: rows that no 16-byte loads fit (70, 99), that lie back to back (50), that 16 bytes fit
@pytest.mark.parametrize("n_ens,neurons,dims,bits", [
    (6, 4096, 70, False), (12, 2048, 99, False), (8, 2048, 50, True), (8, 2048, 64, True),
    (2, 7000, 3, False)])
def test_spikes_are_bits_only_where_the_launch_writes_bits(queue, n_ens, neurons, dims, bits):
    """Spikes that nothing but launches visiting active columns reads."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        net = mb.Network(seed=3, solver="surrogate")
        stim = net.Node(mb.WhiteSignal(period=0.5, high=6.0, seed=3), size_out=dims)
        ens = [net.Ensemble(neurons, dims) for _ in range(n_ens)]
        for k in range(n_ens):
            net.Connection(stim, ens[k], synapse=mb.Lowpass(0.005))
            net.Connection(ens[k], ens[k - 1], synapse=mb.Lowpass(0.005))
        return net, net.Probe(ens[0], synapse=0.01)

    (net, probe), (net_o, probe_o) = make(), make()
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        assert any(getattr(p, "event_driven", False) for p in gpu._plans)
        gpu.run_steps(30)
        cpu.run_steps(30)
        assert np.any(gpu.data[probe] != 0) and np.array_equal(gpu.data[probe], cpu.data[probe_o])
        assert np.array_equal(gpu.signal_buffer(), cpu.signal_buffer())
        assert bool(gpu._spike_bits) == bits


@pytest.mark.parametrize("what", ["conv", "long rows", "group per row", "oja", "voja", "bcm"])
def test_infinities_and_nan_reach_the_results_they_reach_in_the_oracle(queue, rng, what):
    from nengo_ocl_amd import hipra_gemv
    from nengo_ocl_amd import hipra_nonlinearities as nl
    from oracle import oracle as orc

    def odd(n, share=0.004):
        v = rng.normal(size=n)
        at = rng.uniform(size=n) < share
        v[at] = rng.choice([np.nan, np.inf, -np.inf, -0.0, np.finfo(np.float32).max], size=at.sum())
        return v

    if what == "conv":
        data = RA([odd(9 * 8 * 16), odd(9 * 16 * 20, 0.001), np.zeros(9 * 8 * 20)])
        run = lambda mod, q, d: [mod.plan_conv2d(q, d[[0]], d[[2]], d[[1]], (9, 8, 16), (9, 8, 20),
                                                 (3, 3), padding="same", channels_last=True)]
    elif what in ("long rows", "group per row"):
        m, n = {"long rows": (90, 700), "group per row": (40, 4100)}[what]
        data = RA([odd(m * n, 1 / 3000).reshape(m, n), odd(n, 1 / 2000), odd(m, 0.05)])
        js = RA([[0]], dtype=np.int32)
        run = lambda mod, q, d: mod.plan_block_gemv(
            q, 1.0, d[[0]], RA([[0]], dtype=np.int32), d[[1]], js, 1.0, d[[2]]).plans
    else:
        data = RA([odd(100), odd(130, 0.05), odd(130 * 100).reshape(130, 100), odd(130), odd(1), odd(130),
                   odd(130 * 100).reshape(130, 100)])
        alpha, beta = np.float32([1e-3]), np.float32([1.5])
        run = lambda mod, q, d: [
            mod.plan_oja(q, d[[0]], d[[1]], d[[2]], d[[6]], alpha, beta, inc=True) if what == "oja" else
            mod.plan_bcm(q, d[[0]], d[[1]], d[[3]], d[[6]], alpha, inc=True) if what == "bcm" else
            mod.plan_voja(q, d[[0]], d[[1]], d[[2]], d[[6]], d[[4]], d[[5]], alpha, inc=True)]
    dev = to_dev(queue, data)
    run_plans(run(nl if what in ("conv", "oja", "voja", "bcm") else hipra_gemv, queue, dev))
    run_plans(run(orc, None, data))
    got, expected = dev.buf, data.buf
    nan = np.isnan(expected)
    assert nan.any() and not nan.all() and np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), expected[~nan].view(np.uint32))


# tasks of the small-item kernel, and of the large-item kernel: rows that lie back to back, four columns,
# rows that no 16-byte loads fit, 16, 64 and 200 columns
@pytest.mark.parametrize("neurons,dims", [(41, 2), (701, 50), (2101, 4), (203, 70), (1000, 16), (300, 64),
                                          (150, 200)])
@pytest.mark.parametrize("kind", ["LIFRate", "AdaptiveLIF", "AdaptiveLIFRate", "RectifiedLinear",
                                  "SpikingRectifiedLinear", "Sigmoid"])
def test_neuron_types_in_the_launch_of_their_currents(queue, kind, neurons, dims):
    """Every neuron type is updated by the launch that encodes its input, which also forms the sums
    of decoded values it encodes; an ensemble that nothing feeds rides along."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        net = mb.Network(seed=6, solver="surrogate")
        stim = net.Node(mb.WhiteSignal(period=0.5, high=6.0, seed=3), size_out=dims)
        kw = dict(neuron_type=getattr(mb, kind)(), radius=2.0)
        a, b, idle = (net.Ensemble(neurons, dims, **kw) for _ in range(3))
        net.Connection(stim, a, synapse=mb.Lowpass(0.005))
        net.Connection(a, b, synapse=mb.Lowpass(0.005))
        net.Connection(idle, b, synapse=mb.Lowpass(0.005))
        net.Connection(b, a, synapse=mb.Lowpass(0.005))
        return net, net.Probe(b, synapse=0.01)

    (net, probe), (net_o, probe_o) = make(), make()
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        names = [p.name for p in gpu._plans]
        assert any(n.endswith("_neuron") for n in names), names
        gpu.run_steps(40)
        cpu.run_steps(40)
        assert np.any(gpu.data[probe] != 0) and np.array_equal(gpu.data[probe], cpu.data[probe_o])
        assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))


# the small-item kernel with four lanes and with a wave or a group per row, the large-item kernel, the
# launch that visits active columns (one and several groups of 64 rows)
@pytest.mark.parametrize("kind,neurons,dims,ensembles,launch", [
    ("LIF", 41, 2, 3, "wave_ref_filter"), ("LIFRate", 2000, 32, 4, "tile_filter"),
    ("LIFRate", 9000, 3, 3, "tile_filter"), ("LIFRate", 701, 64, 40, "tile_filter"),
    ("LIFRate", 150, 200, 3, None), ("LIF", 1501, 50, 3, "events_filter"),
    ("LIF", 5000, 130, 3, "events_filter"), ("LIF", 1024, 32, 48, "events_filter")])
def test_filters_of_second_order_in_the_launch_of_their_input(queue, kind, neurons, dims, ensembles, launch):
    """Every synapse with at most two coefficients on a side is stepped by the launch that decodes
    its input, several of one decoded value included; one of third order keeps its launch."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    synapses = [mb.Alpha(0.01), mb.LinearFilter([0.3, 0.2], [1.0, -0.5], analog=False),
                mb.LinearFilter([0.4], [1.0, -0.7, 0.2], analog=False), mb.Lowpass(0.005),
                mb.LinearFilter([0.4, 0.1], [1.0], analog=False),
                mb.LinearFilter([0.1], [1.0, -0.7, 0.2, 0.1], analog=False)]

    def make():
        net = mb.Network(seed=6, solver="surrogate", share_decoded=True)
        stim = net.Node(mb.WhiteSignal(period=0.5, high=6.0, seed=3), size_out=dims)
        ens = [net.Ensemble(neurons, dims, neuron_type=getattr(mb, kind)(), radius=2.0)
               for _ in range(ensembles)]
        net.Connection(stim, ens[0], synapse=mb.Alpha(0.005))
        for k in range(ensembles):
            for u, synapse in enumerate(synapses if k == 0 else synapses[k % 5:k % 5 + 1]):
                net.Connection(ens[k], ens[(k + u + 1) % ensembles], synapse=synapse, transform=0.3)
        return net, [net.Probe(ens[1], synapse=mb.Alpha(0.01)), net.Probe(ens[-1], synapse=0.01)]

    (net, probes), (net_o, probes_o) = make(), make()
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        cpu.run_steps(40)
        names = [p.name for p in gpu._plans]
        fused = [p for p in gpu._plans if getattr(p, "filter_state", None) is not None]
        assert fused and (launch is None or any(p.name == "hipra_gemv." + launch for p in fused)), names
        for _ in range(2):  # the second time from a reset: the filters' states with it
            gpu.run_steps(40)
            for p, p_o in zip(probes, probes_o):
                assert np.any(gpu.data[p] != 0) and np.array_equal(gpu.data[p], cpu.data[p_o])
            assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))
            gpu.reset()


# waves of sixteen rows and of 64, populations that end inside a wave and inside a word; columns on both
# sides of 65,536, whole slices (120,000 and 140,000 rows), more columns than 17 bits hold, as many bits as
# the LDS holds and one more
@pytest.mark.parametrize("n,fan_out,lead,bits", [
    (65, 30, 0, True), (2001, 40, 0, True), (1000, 30, 48, True), (1000, 30, 50, False), (33000, 60, 0, True),
    (70001, 30, 0, True), (120000, 15, 0, True), (140000, 14, 0, True), (1179520, 2, 0, True),
    (1179521, 2, 0, False)])
def test_sparse_products_read_the_bits_their_neurons_left(queue, n, fan_out, lead, bits):
    """A population's spikes reach the sparse products that read them as bits from the launch that
    updates the neurons (not where another population's rows (`lead`) leave them inside a wave), and
    the spikes the host sees stay floats that it may write."""
    from nengo_ocl_amd import configs
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        rng = np.random.RandomState(4)
        net = mb.Network(seed=2)
        first = net.Ensemble(lead, 1, neuron_type=mb.LIF(tau_ref=0.001)) if lead else None
        ens = net.Ensemble(n, 1, neuron_type=mb.LIF(tau_ref=0.001, amplitude=0.7))
        if lead:  # both in one launch
            stim = net.Node(mb.WhiteSignal(period=0.5, high=6.0, seed=3), size_out=1)
            for e in (first, ens):
                net.Connection(stim, e, synapse=mb.Lowpass(0.005))
        for _ in range(2):  # two products of the same spikes
            weights = configs.sparse_ring_weights(n, fan_out, 0.3, rng, scale=2e-4)
            net.Connection(ens.neurons, ens.neurons, transform=mb.Sparse((n, n), weights),
                           synapse=mb.Lowpass(0.05))
        return net, [net.Probe(e.neurons, synapse=0.01) for e in (first, ens) if e is not None]

    (net, probes), (net_o, probes_o) = make(), make()
    with Simulator(net, seed=1, event_calibration_steps=0) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        names = [getattr(p.kern, "__name__", "") for p in gpu._plans]
        assert ("nhip_spmv_sell_bits" in names) == bits, names
        for _ in range(2):
            gpu.run_steps(15)
            cpu.run_steps(15)
            for p, p_o in zip(probes, probes_o):
                assert np.any(gpu.data[p] != 0) and np.array_equal(gpu.data[p], cpu.data[p_o])
            assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))
            for sim in (gpu, cpu):  # what the host puts there is replaced before the product reads it
                spikes = next(op.output for op in sim.operators if type(op).__name__ == "SimNeurons"
                              and op.output.size == n)
                sim.signals[spikes] = np.ones(spikes.shape)


# rows of one tile, of a partial one, of whole passes of 2048 columns and a bit more, on 16-byte boundaries
# and not; groups that end inside their four rows; an infinite and a NaN weight
@pytest.mark.parametrize("n_pre,n_post", [(4, 3), (50, 60), (301, 90), (128, 1000), (1000, 129), (2048, 66),
                                          (2049, 70), (2500, 101), (4100, 33)])
@pytest.mark.parametrize("rule", ["Oja", "BCM"])
@pytest.mark.parametrize("odd", [False, True])
def test_rules_between_neurons_in_the_launch_of_their_product(queue, rule, n_pre, n_post, odd):
    """A matrix that Oja's or the BCM rule changes is read once per step: by the launch that multiplies
    by it, which also steps the filters of its product and of the activities the rule reads."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        rng = np.random.RandomState(8)
        net = mb.Network(seed=5, solver="surrogate")
        stim = net.Node(mb.WhiteSignal(period=0.5, high=6.0, seed=3), size_out=2)
        pre, post = net.Ensemble(n_pre, 2), net.Ensemble(n_post, 2)
        net.Connection(stim, pre, synapse=mb.Lowpass(0.005))
        learning = mb.Oja(learning_rate=1e-4, beta=0.7) if rule == "Oja" else mb.BCM(learning_rate=1e-7)
        synapses = [mb.Lowpass(0.005), mb.Alpha(0.01)] if odd else [mb.Lowpass(0.005)]
        for synapse in synapses:  # two learned matrices with the same activities
            weights = rng.normal(scale=1e-1 / n_pre, size=(n_post, n_pre))
            if odd:
                weights[n_post // 2, n_pre // 3], weights[1, 0] = np.inf, np.nan
            net.Connection(pre.neurons, post.neurons, transform=weights, learning_rule=learning, synapse=synapse)
            learning = mb.Oja(learning_rate=1e-4) if rule == "Oja" else mb.BCM(learning_rate=1e-7)
        return net, [net.Probe(post, synapse=0.01)]

    (net, probes), (net_o, probes_o) = make(), make()
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        launches = [getattr(p, "kern").__name__ for p in gpu._plans if hasattr(p, "kern")]
        assert "nhip_gemv_learn" in launches and "nhip_learning_rule" not in launches, launches
        if not odd:
            assert not {"nhip_linearfilter", "nhip_sequence_chains"} & set(launches), launches
        for _ in range(2):
            gpu.run_steps(20)
            cpu.run_steps(20)
            got, want = gpu.signal_buffer(), cpu.signal_buffer()
            nan = np.isnan(want)
            assert np.array_equal(np.isnan(got), nan) and nan.any() == odd
            assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
            for p, p_o in zip(probes, probes_o):
                assert np.array_equal(gpu.data[p], cpu.data[p_o], equal_nan=True)


# fewer columns than a quad and one behind it, one group more than there are counters of arrivals, an odd
# remainder behind a whole pass
@pytest.mark.parametrize("n_pre,n_post", [(1, 5), (2, 9), (3, 129), (5, 133), (2051, 7)])
@pytest.mark.parametrize("rule", ["Oja", "BCM"])
def test_learned_rows_that_do_not_end_with_a_quad(queue, rule, n_pre, n_post):
    test_rules_between_neurons_in_the_launch_of_their_product(queue, rule, n_pre, n_post, False)


@pytest.mark.parametrize("rule", ["Oja", "BCM"])
@pytest.mark.parametrize("rows,cols", [(slice(0, 150), slice(None)), (slice(None), slice(20, 200)),
                                       (slice(7, 8), slice(None))])
def test_products_with_a_part_of_a_learned_matrix_read_it_unchanged(queue, rule, rows, cols):
    """Another product of the step reads some rows or columns of the matrix that the rule changes."""
    from nengo_ocl_amd import ir
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    rng = np.random.RandomState(8)
    net = mb.Network(seed=5, solver="surrogate")
    stim = net.Node(mb.WhiteSignal(period=0.5, high=6.0, seed=3), size_out=2)
    pre, post = net.Ensemble(300, 2), net.Ensemble(300, 2)
    net.Connection(stim, pre, synapse=mb.Lowpass(0.005))
    learning = mb.Oja(learning_rate=1e-4, beta=0.7) if rule == "Oja" else mb.BCM(learning_rate=1e-7)
    net.Connection(pre.neurons, post.neurons, transform=rng.normal(scale=1e-3, size=(300, 300)),
                   learning_rule=learning, synapse=mb.Lowpass(0.005))
    model = net.build_model()
    weights = next(op.dst for op in model.operators if isinstance(op, ir.Copy) and op.inc
                   and op.dst.shape == (300, 300))
    x = next(op.X for op in model.operators if isinstance(op, ir.DotInc) and op.A is weights)
    part = weights[rows, cols]
    y = ir.Signal(np.zeros(part.shape[0]), name="a part of the product")
    model.add_op(ir.Reset(y))
    model.add_op(ir.DotInc(part, x[cols], y))
    with Simulator(None, model=model, seed=1) as gpu, OracleSimulator(None, model=model, seed=1) as cpu:
        for _ in range(3):
            gpu.run_steps(20)
            cpu.run_steps(20)
            assert np.any(cpu.signals[y] != 0)
            assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))


@pytest.mark.parametrize("rule", ["Oja", "BCM"])
@pytest.mark.parametrize("n,extra,synapses", [
    (300, [(2300, 2)], ["Lowpass"]), (300, [(3701, 64)], ["Lowpass"]), (50, [(20, 50)] * 115, ["Lowpass", "Alpha"]),
    (301, [(3700, 63), (3, 301)], ["Alpha"]), (300, [(2301, 3), (1024, 64)], ["Lowpass", "Alpha"]),
    (300, [(17200, 512), (40, 1024)], ["Lowpass", "Alpha"])])
def test_products_apart_from_the_launch_of_learned_matrices(queue, rule, n, extra, synapses):
    """Too many other products for that launch: they keep their filters, of first and second order, in a launch
    in front of it."""
    from test_launch_rules import rule_beside_products
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    nets = [rule_beside_products(n, extra, rule, synapses) for _ in range(2)]
    with Simulator(nets[0], seed=1, event_calibration_steps=0) as gpu, OracleSimulator(nets[1], seed=1) as cpu:
        learn = next(k for k, p in enumerate(gpu._plans) if getattr(p, "learned_matrices", 0))
        assert any(p.name.endswith("_filter") for p in list(gpu._plans)[:learn])
        cpu.run_steps(30)
        for _ in range(2):  # the second time from a reset: the filters' states with it
            gpu.run_steps(30)
            assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))
            gpu.reset()


@pytest.mark.parametrize("synapse", ["Alpha", "third order"])
@pytest.mark.parametrize("n,dims", [(200, 2), (512, 32), (1031, 3)])
def test_synapses_of_every_order_beside_learned_decoders(queue, synapse, n, dims):
    """The launch of a step's synapses is taken apart: some ride in a product's launch, the activities' in that
    of the weights, the others keep one; from the start and from a reset."""
    from test_launch_rules import pes_with_synapses
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    nets = [pes_with_synapses(synapse, n, dims) for _ in range(2)]
    with Simulator(nets[0], seed=1, event_calibration_steps=0) as gpu, OracleSimulator(nets[1], seed=1) as cpu:
        cpu.run_steps(40)
        for _ in range(2):
            gpu.run_steps(40)
            for p, p_o in zip(nets[0].probes, nets[1].probes):
                assert np.array_equal(gpu.data[p], cpu.data[p_o])
            assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))
            gpu.reset()


@pytest.mark.parametrize("kind,neurons,dims,ensembles", [
    ("LIF", 100, 1, 2), ("LIF", 30, 1, 2), ("LIF", 65, 3, 5), ("LIFRate", 33, 2, 4), ("AdaptiveLIF", 40, 1, 9),
    ("RectifiedLinear", 17, 4, 3), ("SpikingRectifiedLinear", 130, 2, 3), ("Sigmoid", 9, 6, 3),
    ("LIF", 300, 4, 3), ("LIF", 7, 2, 5), ("LIFRate", 260, 1, 2), ("LIF", 129, 12, 2)])
def test_small_networks_run_resident(queue, monkeypatch, kind, neurons, dims, ensembles):
    """Networks that fit the LDS of a compute unit take all steps of a call in one launch: first- and
    second-order synapses, sums of inputs, function and table nodes, probes with a period; calls of
    one and of several steps, a reset between them."""
    from nengo_ocl_amd import hipra_resident
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        net = mb.Network(seed=6, solver="surrogate")
        stim = net.Node(mb.WhiteSignal(period=0.05, high=60.0, seed=3), size_out=dims)
        wave = net.Node(np.sin)
        ens = [net.Ensemble(neurons, dims, neuron_type=getattr(mb, kind)(), radius=2.0) for _ in range(ensembles)]
        net.Connection(stim, ens[0], synapse=mb.Alpha(0.005))
        net.Connection(wave, ens[1], transform=np.ones((dims, 1)), synapse=mb.Lowpass(0.01))
        for k in range(ensembles):
            for u, synapse in enumerate((mb.Lowpass(0.005), mb.Alpha(0.01))):
                net.Connection(ens[k], ens[(k + u + 1) % ensembles], synapse=synapse, transform=0.6)
        probes = [net.Probe(ens[1], synapse=mb.Alpha(0.01)), net.Probe(ens[-1], synapse=0.01, sample_every=0.003),
                  net.Probe(ens[0].neurons), net.Probe(wave)]
        return net, probes

    monkeypatch.setattr(hipra_resident, "GRAPH_LAUNCH", 1e9)  # also where a graph would be shorter
    (net, probes), (net_o, probes_o) = make(), make()
    with Simulator(net, seed=1, n_prealloc_probes=32) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        assert gpu._plans.resident is not None, [p.name for p in gpu._plans]
        for repeat in range(2):
            for n in (1, 2, 37, 1, 64):
                gpu.run_steps(n)
                if repeat == 0:
                    cpu.run_steps(n)
                    assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32)), n
            for p, p_o in zip(probes, probes_o):
                assert np.any(gpu.data[p] != 0) and np.array_equal(gpu.data[p], cpu.data[p_o])
            assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))
            gpu.reset()


# the tiled kernel and the one of a wave per group; layers of every kind of epilogue
@pytest.mark.parametrize("kind", ["RectifiedLinear", "LIF", "AdaptiveLIF", "LIFRate", "Sigmoid",
                                  "SpikingRectifiedLinear", "AdaptiveLIFRate"])
@pytest.mark.parametrize("size,channels,filters,synapse", [(12, 1, 5, "lowpass"), (17, 3, 16, "alpha"),
                                                           (26, 2, 32, "lowpass")])
def test_convolutions_update_the_neurons_and_filters_they_feed(queue, kind, size, channels, filters, synapse):
    """A layer's neurons are updated by the convolution that forms their currents, the synapse behind a
    convolution is stepped by it, and nothing resets what it overwrites; the image and the samples of a large
    layer ride in another launch."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        rng = np.random.RandomState(3)
        net = mb.Network(seed=7, solver="surrogate")
        kw = dict(neuron_type=getattr(mb, kind)(), max_rates=(100, 200), intercepts=(-0.5, 0.5))
        eye = net.Node(mb.PresentInput(rng.uniform(size=(3, size * size * channels)), 0.004),
                       size_out=size * size * channels)
        first = mb.Convolution(filters, (size, size, channels), kernel_size=(3, 3), seed=1)
        second = mb.Convolution(2 * filters, tuple(first.spec.output_shape.shape), kernel_size=(3, 3),
                                strides=(2, 2), seed=2,
                                init=rng.uniform(-1, 1, size=(3, 3, filters, 2 * filters)) / (9.0 * filters))
        layers = [net.Ensemble(c.size_out, 1, encoders=np.ones((c.size_out, 1)), **kw) for c in (first, second)]
        net.Connection(eye, layers[0].neurons, transform=first, synapse=None)
        net.Connection(layers[0].neurons, layers[1].neurons, transform=second,
                       synapse=mb.Alpha(0.003) if synapse == "alpha" else mb.Lowpass(0.005))
        out = net.Node(None, size_in=3)
        net.Connection(layers[1].neurons, out, synapse=mb.Lowpass(0.005),
                       transform=rng.normal(scale=1e-2 / second.size_out, size=(3, second.size_out)))
        return net, [net.Probe(out), net.Probe(layers[1].neurons, sample_every=0.004), net.Probe(layers[0].neurons)]

    (net, probes), (net_o, probes_o) = make(), make()
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        cpu.run_steps(25)
        launches = [p.kern.__name__ for p in gpu._plans]
        assert {"nhip_conv2d_neuron", "nhip_conv2d_filter"} <= set(launches), launches
        assert not {"nhip_conv2d", "nhip_reset", "nhip_linearfilter"} & set(launches), launches
        for _ in range(2):
            gpu.run_steps(25)
            assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))
            for p, p_o in zip(probes, probes_o):
                assert np.any(gpu.data[p] != 0) and np.array_equal(gpu.data[p], cpu.data[p_o])
            gpu.reset()


# rows on both sides of the limit for a lane per row; neurons around the 64 rows of a task
@pytest.mark.parametrize("kind", ["LIF", "LIFRate"])
@pytest.mark.parametrize("n_ens,neurons,parts,lanes", [(48, 64, 3, 64), (46, 65, 3, 4), (40, 103, 70, 64),
                                                       (333, 13, 4, 64), (70, 60, 2, 4)])
def test_waves_form_the_sums_of_many_inputs(queue, kind, n_ens, neurons, parts, lanes):
    """Neurons in one launch with the sums of their inputs, one to three dimensions, and a sum that no
    neuron reads."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        rng = np.random.RandomState(n_ens)
        net = mb.Network(seed=2, solver="surrogate")
        ens = [net.Ensemble(neurons, 1 + i % 3, neuron_type=getattr(mb, kind)()) for i in range(n_ens)]
        out = net.Node(None, size_in=2)
        for i, e in enumerate(ens):
            for j in rng.choice(n_ens, size=parts, replace=parts > n_ens):
                net.Connection(ens[j], e, synapse=mb.Lowpass(0.005), transform=rng.uniform(
                    -1, 1, size=(1 + i % 3, 1 + int(j) % 3)))
        for e in ens[:9:3]:
            net.Connection(e, out, synapse=mb.Lowpass(0.005), transform=rng.normal(size=(2, 1)))
        return net, net.Probe(out)

    (net, probe), (net_o, probe_o) = make(), make()
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        fused = [p for p in gpu._plans if getattr(p, "input_sums", 0)]
        assert len(fused) == 1 and fused[0].args[0] == lanes, [(p, p.args[0]) for p in fused]
        cpu.run_steps(20)
        gpu.run_steps(20)
        assert np.array_equal(gpu.signal_buffer().view(np.uint32), cpu.signal_buffer().view(np.uint32))
        assert np.any(gpu.data[probe] != 0) and np.array_equal(gpu.data[probe], cpu.data[probe_o])
