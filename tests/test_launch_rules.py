"""Which kernel a launch takes, by its sizes: rules that can be followed without a device."""

import numpy as np
import pytest

from helpers import RA, host_queue, host_simulators, to_dev


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


def learned_products(queue, rule, unlearned=(), learned=((0, 300, 300),), aliases=()):
    """`hipra_gemv.fuse_hebbian` for products with matrices of the rule (`learned`: offset in the matrix
    buffer, rows, columns) and with others (`unlearned`: the same, or (None, rows, columns) for one of its
    own); `aliases`: operand ("x", "pre", "post", "y_in") -> its offset in the matrix buffer."""
    from nengo_ocl_amd import hipra_gemv, hipra_nonlinearities as nl
    from nengo_ocl_amd.hipraggedarray import HIPRaggedArray

    aliases, items = dict(aliases), list(learned) + list(unlearned)
    host = RA([np.zeros((300, 400))] + [np.zeros(n) for n in (5000, 5000, 5000)]
              + [np.zeros((m, n)) for at, m, n in items if at is None] + [np.zeros(m) for _, m, _ in items])
    dev = to_dev(queue, host)
    own = iter(range(4, len(host)))
    starts = [next(own) if at is None else None for at, _, _ in items]
    outs = [int(host.starts[next(own)]) for _ in items]

    def view(start, m, n, stride=None):
        one = lambda v: np.array([v], dtype=np.int32)
        return HIPRaggedArray.from_buffer(queue, dev.dev_buf, one(start), one(m), one(n), one(stride or n), one(1))

    def column(what, k, n):
        return view(aliases.get(what, int(host.starts[k])), n, 1)

    cat = hipra_gemv._concat
    matrix = [view(at if at is not None else int(host.starts[s]), m, n, 400 if at is not None else n)
              for (at, m, n), s in zip(items, starts)]
    A = cat(matrix)
    X = cat([column("x" if k else "", 1, n) for k, (_, _, n) in enumerate(items)])
    Y = cat([view(out, m, 1) for out, (_, m, _) in zip(outs, items)])
    Y_in = cat([column("y_in", 3, m) if "y_in" in aliases and k == len(items) - 1 else view(out, m, 1)
                for k, (out, (_, m, _)) in enumerate(zip(outs, items))])
    js = RA([[k] for k in range(len(items))], dtype=np.int32)
    prog = hipra_gemv.plan_block_gemv(queue, 1.0, A, js, X, js, 0.0, Y, Y_in=Y_in)
    pre = cat([column("pre", 1, n) for _, _, n in learned])
    post = cat([column("post", 2, m) for _, m, _ in learned])
    delta, ones = cat(matrix[:len(learned)]), np.ones(len(learned), dtype=np.float32)
    plan = (nl.plan_oja(queue, pre, post, delta, delta, ones, ones, inc=True) if rule == "Oja" else
            nl.plan_bcm(queue, pre, post, cat([column("theta", 3, m) for _, m, _ in learned]), delta, ones, inc=True))
    return prog.plans, hipra_gemv.fuse_hebbian(prog.plans, plan)


# other rows, other columns and the inside of the learned matrix (300 rows, 400 apart), one row of it, a row
# that starts behind its columns; vectors and an old output that lie in it; rules of two overlapping matrices
@pytest.mark.parametrize("rule", ["Oja", "BCM"])
@pytest.mark.parametrize("unlearned,learned,aliases,fused", [
    ((), [(0, 300, 300)], {}, True),
    ([(None, 200, 300)], [(0, 300, 300)], {}, True),
    ([(None, 200, 300)], [(0, 150, 300), (150 * 400, 150, 300)], {}, True),
    ([(0, 150, 300)], [(0, 300, 300)], {}, False),
    ([(0, 300, 200)], [(0, 300, 300)], {}, False),
    ([(100 * 400 + 100, 150, 200)], [(0, 300, 300)], {}, False),
    ([(299 * 400, 1, 300)], [(0, 300, 300)], {}, False),
    ([(149 * 400 + 300, 1, 200)], [(0, 150, 300)], {}, True),
    ([(None, 200, 300)], [(0, 300, 300)], {"x": 400}, False),
    ([(None, 200, 300)], [(0, 300, 300)], {"y_in": 400}, False),
    ((), [(0, 300, 300)], {"pre": 50 * 400}, False),
    ((), [(0, 300, 300)], {"post": 50 * 400}, False),
    ((), [(0, 151, 300), (150 * 400, 150, 300)], {}, False)])
def test_learned_matrices_are_not_written_where_their_launch_reads(monkeypatch, rule, unlearned, learned, aliases,
                                                                   fused):
    _, result = learned_products(host_queue(monkeypatch), rule, unlearned, learned, aliases)
    assert (result is not None) == fused


@pytest.mark.parametrize("rows,fused", [(None, True), (slice(0, 16), False), (slice(31, 32), False),
                                        (slice(None), False)])
def test_learned_decoders_are_not_written_where_their_launch_reads(monkeypatch, rows, fused):
    """The same for decoders learned from an error signal: a second product with some of their rows or with
    all of them, of other activities."""
    from nengo_ocl_amd import configs, ir
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    model = configs.c4_pes(1, n_triples=4, n_neurons=1024, dims=32)[0].build_model()
    if rows is not None:
        learned = [op.dst for op in model.operators if isinstance(op, ir.Copy) and op.inc
                   and op.dst.shape == (32, 1024)]
        x = next(op.X for op in model.operators if isinstance(op, ir.DotInc) and op.A is learned[1])
        y = ir.Signal(np.zeros(len(range(32)[rows])), name="part")
        model.add_op(ir.Reset(y))
        model.add_op(ir.DotInc(learned[0][rows], x, y))
    with Simulator(None, model=model, seed=1, event_calibration_steps=0) as sim:
        assert max(getattr(p, "learned_matrices", 0) for p in sim._plans) == (4 if fused else 0)


@pytest.mark.parametrize("n_cols,bits", [(1179520, True), (1179521, False), (1179648, False)])
def test_spikes_are_handed_on_as_bits_where_the_product_holds_them(monkeypatch, n_cols, bits):
    """On both sides of the longest X of the launch that is handed bits (nhip_spmv_sell_bits refuses longer
    ones), up to the longest of the one that forms them."""
    import scipy.sparse
    from nengo_ocl_amd import hipra_spmv, minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setattr(hipra_spmv, "SKIP_MIN_WIDTH", 0)  # (nearly all rows are empty)
    net = mb.Network(seed=1, solver="surrogate")
    ens = net.Ensemble(n_cols, 1)
    weights = scipy.sparse.csr_matrix((np.ones(320), (np.repeat(np.arange(10), 32), np.arange(320) * 3600)),
                                      shape=(n_cols, n_cols))
    net.Connection(ens.neurons, ens.neurons, transform=mb.Sparse((n_cols, n_cols), weights),
                   synapse=mb.Lowpass(0.01))
    with Simulator(net, seed=1, event_calibration_steps=0) as sim:
        kerns = [p.kern.__name__ for p in sim._plans]
    assert ("nhip_spmv_sell_bits" in kerns) == ("nhip_gemv_rows_lif_bits" in kerns) == bits, kerns
    assert bits or "nhip_spmv_sell_spikes" in kerns


@pytest.mark.parametrize("synapse", ["Alpha", "Lowpass"])
def test_one_copy_of_a_sparse_matrix_stays_on_the_device(monkeypatch, synapse):
    """A product that is handed bits keeps its own layout of the matrix and gives the other one back."""
    import gc
    import weakref

    from nengo_ocl_amd import configs, hipra_spmv, minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    made, upload = [], hipra_spmv.to_device

    def to_device(queue, array):
        made.append(upload(queue, array))
        return made[-1]

    monkeypatch.setattr(hipra_spmv, "to_device", to_device)
    net = mb.Network(seed=1)
    ens = net.Ensemble(2001, 1)
    weights = configs.sparse_ring_weights(2001, 40, 0.3, np.random.RandomState(4), scale=2e-4)
    net.Connection(ens.neurons, ens.neurons, transform=mb.Sparse((2001, 2001), weights),
                   synapse=getattr(mb, synapse)(0.01))
    with Simulator(net, seed=1, event_calibration_steps=0) as sim:
        product, = [p for p in sim._plans if p.kern.__name__ == "nhip_spmv_sell_bits"]
        made = [weakref.ref(a) for a in made]
        gc.collect()
        alive = [r() for r in made if r() is not None]
        assert alive and len(alive) < len(made)
        assert all(any(a is kept for kept in product.full_args) for a in alive)


# words before, inside and behind an array of 32 words at word 64
@pytest.mark.parametrize("first,words,where", [(64, 32, 0), (72, 8, 8), (88, 8, 24), (32, 32, 32), (96, 4, 32),
                                               (60, 8, None), (32, 33, None), (60, 100, None), (92, 8, None),
                                               (88, 9, None)])
def test_arrays_of_a_resident_network_have_one_copy(first, words, where):
    """An array inside another one is found there, one that reaches over its start or end is refused."""
    from nengo_ocl_amd import hipra_resident

    image = hipra_resident._Image(None)
    assert image.add(4 * 64, 32) == 0
    if where is None:
        with pytest.raises(hipra_resident._Unfit):
            image.add(4 * first, words)
    else:
        assert image.add(4 * first, words) == where


def rule_beside_products(n, extra, rule="Oja", synapses=("Lowpass",)):
    """Two populations of n neurons with a learned matrix between them; `extra`: (rows, neurons) of products
    of other populations in the same step."""
    from nengo_ocl_amd import minibuilder as mb

    rng = np.random.RandomState(1)
    net = mb.Network(seed=5, solver="surrogate")
    stim = net.Node(mb.WhiteSignal(period=0.5, high=6.0, seed=3), size_out=2)
    pre, post = net.Ensemble(n, 2), net.Ensemble(n, 2)
    net.Connection(stim, pre, synapse=mb.Lowpass(0.005))
    learning = mb.Oja(learning_rate=1e-6, beta=0.7) if rule == "Oja" else mb.BCM(learning_rate=1e-9)
    net.Connection(pre.neurons, post.neurons, transform=rng.normal(scale=1e-1 / n, size=(n, n)),
                   learning_rule=learning, synapse=mb.Lowpass(0.005))
    for k, (rows, cols) in enumerate(extra):
        other = net.Ensemble(cols, 2)
        net.Connection(stim, other, synapse=mb.Lowpass(0.005))
        net.Connection(other.neurons, net.Node(None, size_in=rows), transform=rng.normal(size=(rows, cols)),
                       synapse=getattr(mb, synapses[k % len(synapses)])(0.005))
    return net


# rows and columns of the others on both sides of what rides along: at most four columns, more, many, and rows
# that no 16-byte loads fit; in the class of the learned matrix (300 x 300, 50 x 50) and in another
@pytest.mark.parametrize("n,extra,rides", [
    (300, [(2180, 2)], True), (300, [(2184, 2)], False), (300, [(3636, 4)], True), (300, [(3640, 4)], False),
    (300, [(100000, 2)], False), (300, [(3636, 64)], True),
    (300, [(3640, 64)], False), (300, [(2, 300)] * 16, True), (300, [(7740, 300)], True),
    (300, [(7744, 300)], False), (50, [(20, 50)] * 109, True), (50, [(20, 50)] * 110, False),
    (301, [(7760, 301)], True), (301, [(7764, 301)], False), (300, [(2184, 2), (3636, 64)], None)])
def test_few_other_products_ride_with_learned_matrices(monkeypatch, n, extra, rides):
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    with Simulator(rule_beside_products(n, extra), seed=1, event_calibration_steps=0) as sim:
        learn, = [p for p in sim._plans if getattr(p, "learned_matrices", 0)]
        at = list(sim._plans).index(learn)
        front = [p for p in list(sim._plans)[:at] if p.name.endswith("_filter")]
    groups = [-(-rows // 4) for rows, _ in extra]
    assert learn.n_tasks == -(-n // 4) + (groups[1] if rides is None else sum(groups) if rides else 0)
    assert len(front) == (0 if rides else 1)


# both sides of the limit: two populations (times beside `resident_program`), many small ones, large ones
@pytest.mark.parametrize("what,neurons,resident", [
    ("pair", 30, True), ("pair", 1000, True), ("pair", 1408, True), ("pair", 1500, False), ("pair", 2000, False),
    ("pair", 2500, False), ("graph", 50, True), ("graph", 150, False)])
def test_networks_run_resident_where_that_is_shorter(monkeypatch, what, neurons, resident):
    from nengo_ocl_amd import configs
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    if what == "pair":
        net = configs.c0_readme(5, n_neurons=neurons)[0]
    else:
        net = configs.c2_watts_strogatz(5, n_ens=16, n_neurons=neurons, n_driven=1)[0]
        net.n_eval_points = 300
    with Simulator(net, seed=1, event_calibration_steps=0) as sim:
        assert (sim._plans.resident is not None) == resident


def pes_with_synapses(synapse, n=512, dims=32):
    """Learned decoders, and a probe with a synapse of second or third order."""
    from nengo_ocl_amd import configs, minibuilder as mb

    net = configs.c4_pes(1, n_triples=2, n_neurons=n, dims=dims)[0]
    if synapse == "Alpha":
        net.Probe(net.ensembles[0].neurons, synapse=mb.Alpha(0.01))
    else:
        net.Probe(net.ensembles[0], synapse=mb.LinearFilter([0.1], [1.0, -0.7, 0.2, 0.1], analog=False))
    return net


# spikes of an ensemble behind a second-order synapse (a short launch, which rides, or a long one), a
# decoded value behind one of third order (which would need a launch)
@pytest.mark.parametrize("synapse,n,dims,fused", [
    ("Alpha", 200, 2, True), ("Alpha", 512, 32, True), ("Alpha", 3000, 2, False), ("third order", 512, 32, False)])
def test_synapses_of_higher_order_leave_the_others_their_launch(monkeypatch, synapse, n, dims, fused):
    """Synapses of every class share a launch; one of higher order in it does not keep the activities' filters
    out of the launch of the weights they change, where it finds another to ride in."""
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    apart, some_filters = [], Simulator._some_filters

    def record(sim, lf, which):
        apart.append(some_filters(sim, lf, which))
        return apart[-1]

    monkeypatch.setattr(Simulator, "_some_filters", record)
    with Simulator(pes_with_synapses(synapse, n, dims), seed=1, event_calibration_steps=0) as sim:
        launches = [p.kern.__name__ for p in sim._plans]
        # (a launch that was tried and not taken leaves nothing behind)
        assert any(apart[0].bufpos is pos for pos in sim._filter_positions) == fused
    assert ("nhip_outer_filter" in launches) == fused and ("nhip_elementwise_inc" in launches) != fused, launches


def test_synapses_that_their_product_reads_leave_the_others_in_its_launch(monkeypatch):
    """Among the synapses of one launch are some whose outputs the products read that feed the others."""
    from nengo_ocl_amd.simulator import Simulator
    from random_networks import random_network

    host_simulators(monkeypatch)
    model = random_network(5, big=True, sliced=False, rich=True)[0].build_model()
    with Simulator(None, model=model, seed=1, event_calibration_steps=0) as sim:
        launches = [p.kern.__name__ for p in sim._plans if hasattr(p, "kern")]
    assert {"nhip_gemv_rows_filter", "nhip_gemv_tile_filter"} <= set(launches), launches


def test_populations_without_input_ride_with_unaligned_matrices(monkeypatch):
    """Rows that lie back to back without 16-byte alignment have an instance of their own: a population without
    input joins it, and the launch forms the input sums of the others."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    net = mb.Network(seed=1, solver="surrogate")
    ens = [net.Ensemble(1501, 50) for _ in range(3)]
    for k in (1, 1, 2):  # (nothing reaches the first)
        net.Connection(ens[0], ens[k], synapse=mb.Lowpass(0.005))
    with Simulator(net, seed=1, event_calibration_steps=0) as sim:
        neurons = [p for p in sim._plans if p.name.endswith("_lif")]
        assert len(neurons) == 1 and neurons[0].input_sums == 2, [p.name for p in sim._plans]


def test_planning_of_many_populations_looks_at_each_a_few_times(monkeypatch):
    """What a launch with input sums must not overlap is looked up for all of its items at once."""
    from nengo_ocl_amd import hipra_gemv, minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    looked_at, overlapping = [0], hipra_gemv._overlapping

    def counted(a, b):
        looked_at[0] += len(a) + len(b)
        return overlapping(a, b)

    monkeypatch.setattr(hipra_gemv, "_overlapping", counted)
    counts = []
    for n in (40, 160):
        net = mb.Network(seed=0, solver="surrogate")
        ens = [net.Ensemble(4, 5) for _ in range(n)]
        for a, b in zip(ens, ens[1:] + ens[:1]):
            net.Connection(a, b, synapse=mb.Lowpass(0.005))
            net.Connection(b, a, synapse=mb.Lowpass(0.01))
        looked_at[0] = 0
        with Simulator(net, seed=1, event_calibration_steps=0) as sim:
            assert any("input sums" in p.tag for p in sim._plans)
        counts.append(looked_at[0])
    assert counts[1] <= 5 * counts[0], counts
