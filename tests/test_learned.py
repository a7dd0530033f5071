"""Decoders that PES changes in the launch that decodes with them and with others (csrc/gemv_learn.hip): whole networks
against the CPU oracle bit for bit (the reference's order of summation), and the kernel alone, where quads, passes,
records and batches of columns have edges, on whole numbers whose sums are exact in any order."""

import numpy as np
import pytest

from helpers import assert_same_signals, host_simulators


def learning_launch(sim):
    plan, = [p for p in sim._plans if getattr(p, "laid_out", None) is not None
             and p.laid_out[0].__name__ == "nhip_gemv_learn_events"]
    return plan


def network(n, dims):
    from nengo_ocl_amd import configs

    net, probes, _ = configs.c4_pes(1, n_triples=2, n_neurons=n, dims=dims, learning_rate=1e-3)
    return net, list(probes.values())


# whole and partial tiles, one to three passes of rows, two of columns
SIZES = [(1024, 32), (1500, 20), (2048, 64), (2052, 32), (4100, 20)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,dims", SIZES)
def test_learned_decoders_and_others_in_one_launch(queue, n, dims):
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    (net, probes), (net_o, probes_o) = (network(n, dims) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        assert learning_launch(gpu).laid_out[1][12] > 0
        for steps in (1, 40):
            gpu.run_steps(steps)
            cpu.run_steps(steps)
            for p, p_o in zip(probes, probes_o):
                assert np.array_equal(gpu.data[p], cpu.data[p_o])
            assert_same_signals(gpu, cpu)


@pytest.mark.gpu
def test_matrices_that_the_host_changes(queue):
    """... to others with an infinity, and back."""
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    (net, _), (net_o, _) = (network(1024, 32) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        plan = learning_launch(gpu)
        base = sorted((b for bases, p in gpu._laid_out if p is plan for b in bases
                       if b not in gpu._shared), key=gpu.all_bases.index)[0]
        for value in (2.5e-3, np.inf, 5e-4):
            for sim in (gpu, cpu):
                sig = sim.all_bases[gpu.all_bases.index(base)]  # (the two lay their signals out in the same order)
                new = np.linspace(-1e-3, 1e-3, 32 * 1024).reshape(32, 1024)
                new[3, 7] = value
                sim.signals[sig] = new
                sim.run_steps(5)
            got, want = gpu.signal_buffer(), cpu.signal_buffer()
            assert np.isnan(want).any() == (value != 2.5e-3)
            assert np.array_equal(got, want, equal_nan=True)


# rows: 16, 32 and 64 lanes, two records; columns: less than a tile and more, one to three passes
@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 70])
@pytest.mark.parametrize("N", [5, 128, 1003, 2049, 4096, 8200])
def test_columns_beside_a_learned_row(queue, M, N):
    """No, some (more of a tile than a batch holds) and all columns with x != 0; a matrix with an infinity."""
    from nengo_ocl_amd import _lib
    from nengo_ocl_amd.hipraggedarray import empty_device, to_device

    rng = np.random.RandomState(M + N)
    lib, bits = queue.lib, lambda v: int(np.float32(v).view(np.int32))
    for share, odd in ((0.0, False), (0.08, False), (0.3, True), (1.0, False)):
        fixed = rng.randint(-4, 5, size=(M, N)).astype(np.float32)
        learned, rows = rng.randint(-4, 5, size=(3, N)).astype(np.float32), 3
        x = (rng.uniform(size=N) < share) * rng.randint(1, 4, size=N).astype(np.float32)
        f, e = (rng.randint(-3, 4, size=k).astype(np.float32) for k in (N, rows))
        if odd:
            fixed[M // 2, N - 1] = np.inf
        y, y_in, old = (rng.randint(-9, 10, size=k).astype(np.float32) for k in (M + rows, M + rows, M))
        parts = [fixed.ravel(), learned.ravel(), x, f, e, y, y_in, old]
        at = np.concatenate([[0], np.cumsum([p.size for p in parts])])
        B = to_device(queue, np.concatenate(parts))
        mp = -(-M // 16) * 16
        target = [int(at[7]), bits(-0.5), bits(2.0), 1]
        items = np.zeros((-(-M // 64), 32), dtype=np.int32)
        for k in range(len(items)):
            items[k, :20] = ([0, mp, min(64, M - 64 * k), N, at[2], at[5], 1, at[6], 1, bits(2.0), bits(0.5), bits(3.0),
                              0, 1, 64 * k, 0] + target)
        task = np.zeros((1, 32), dtype=np.int32)
        task[0, :24] = [at[1], N, N, at[2], at[5] + M, 1, at[6] + M, 1, bits(1.0), bits(1.0), bits(0.0), 0, rows, 1, 0, 0,
                        16, at[3], at[4], 1, 0, 0, bits(0.5), 0]
        dev = [to_device(queue, a) for a in (task, items, np.array([target], dtype=np.int32),
                                             np.array([[0, N, M, N, 0, mp, 0, len(items)]], dtype=np.int32))]
        columns = empty_device(queue, N * mp)
        _lib.check(lib.nhip_lay_out_columns(queue.handle, dev[3].ptr, 1, N, B.ptr, columns.ptr, dev[1].ptr), "")
        _lib.check(lib.nhip_gemv_learn_events(queue.handle, dev[0].ptr, 1, B.ptr, B.ptr, B.ptr, B.ptr, dev[2].ptr, B.ptr,
                                              None, 0, None, dev[1].ptr, len(items), columns.ptr), "")
        got = np.split(np.asarray(B.get()), at[1:-1])
        with np.errstate(invalid="ignore"):
            want = 2 * (fixed.astype(np.float64) @ x) + 0.5 * y_in[:M] + 3
        assert np.array_equal(got[5][:M], want.astype(np.float32), equal_nan=True), (share, odd)
        assert np.array_equal(got[7], (2 * want + 0.5 * old).astype(np.float32), equal_nan=True)
        assert np.array_equal(got[5][M:], (learned @ x + y_in[M:]).astype(np.float32))
        assert np.array_equal(got[1].reshape(rows, N), learned + 0.5 * np.outer(e, f))


@pytest.mark.parametrize("n,dims", SIZES)
def test_records_cover_every_row_once(monkeypatch, n, dims):
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    with Simulator(network(n, dims)[0], seed=1) as sim:
        plan = learning_launch(sim)
        tasks, records = plan.host_learned
        assert len(tasks) == plan.laid_out[1][1] and len(records) == plan.laid_out[1][12]
        covered = [y + (r + k) * s for y, s, r, c in tasks[:, [4, 5, 11, 12]].tolist() for k in range(c)]
        covered += [y + (r + k) * s for y, s, r, c in records[:, [5, 6, 14, 2]].tolist() for k in range(c)]
        assert sorted(covered) == sorted(
            g["y_start"] + r * g["y_stride0"] for g in (plan.prog.geometry[b] for b in plan.members)
            for r in range(g["y_len"]))
        assert tasks[:, 12].max() <= 4 and records[:, 2].max() <= 64 and not (records[:, 1] % 16).any()


# rows that are read whole beside learned ones, no quad at the end, few groups to an item and one
@pytest.mark.gpu
@pytest.mark.parametrize("n,dims,triples", [(330, 36, 1), (513, 3, 4), (1050, 19, 3), (1028, 7, 5), (2999, 66, 2), (4099, 1, 2)])
def test_activities_replaced_by_their_last_reader(queue, n, dims, triples):
    """Filters of activities that few groups read are stepped by the last of these, in the launch that read them."""
    from nengo_ocl_amd import configs
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    (net, probes, _), (net_o, probes_o, _) = (
        configs.c4_pes(1, n_triples=triples, n_neurons=n, dims=dims, learning_rate=1e-3) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        plan, = [p for p in gpu._plans if getattr(p, "host_learn", None) is not None]
        own = plan.host_learn[0][:, 28:30]
        assert sorted(set(own[own[:, 0] > 0, 1].tolist())) == list(range(triples))
        for steps in (1, 20, 37):
            gpu.run_steps(steps)
            cpu.run_steps(steps)
            for key in probes:
                assert np.array_equal(gpu.data[probes[key]], cpu.data[probes_o[key]])
            assert_same_signals(gpu, cpu)


def rules_on_one_activity(rows, shared, n=1050, dims=20):
    """A decoder learned from the filtered activities of a population, and a matrix of `rows` rows learned from some of
    the same: `shared` "part", the first 700 of them, "all" or "rows", all of them as the column operand of the rule
    and `rows` of them as its row operand too."""
    from nengo_ocl_amd import configs, ir

    net, probes, _ = configs.c4_pes(1, n_triples=1, n_neurons=n, dims=dims, learning_rate=1e-3)
    model = net.build_model(dt=0.001)
    rule, = [op for op in model.operators if isinstance(op, ir.SimPES)]
    spikes, = [op.input for op in model.operators if isinstance(op, ir.SimProcess) and op.output is rule.pre_filtered]
    pre, acts = (rule.pre_filtered[:700], spikes[:700]) if shared == "part" else (rule.pre_filtered, spikes)
    rng = np.random.RandomState(rows)
    weights = ir.Signal(rng.normal(scale=1e-3, size=(rows, pre.size)), name="more.weights")
    delta = ir.Signal(np.zeros(weights.shape), name="more.Delta")
    out = ir.Signal(np.zeros(rows), name="more.out")
    error = (rule.pre_filtered[:rows] if shared == "rows" else
             ir.Signal(rng.normal(size=rows), name="more.error", readonly=True))
    for op in (ir.Reset(out), ir.DotInc(weights, acts, out), ir.SimPES(pre, error, delta, 1e-3),
               ir.Copy(delta, weights, inc=True)):
        model.add_op(op)
    return model, probes


SHARED = [("part", False), ("rows", False), ("all", True)]


@pytest.mark.parametrize("shared,moves", SHARED)
def test_activities_that_others_read_too_are_replaced_behind_the_launch(monkeypatch, shared, moves):
    """The last reader of a filter's output replaces it in the launch only where all readers there read all of it, as
    the rules' column operand: the readers of anything else are not counted."""
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    with Simulator(None, model=rules_on_one_activity(64, shared)[0], seed=1) as sim:
        plan, = [p for p in sim._plans if getattr(p, "host_learn", None) is not None]
        tasks = plan.host_learn[0]
        learned = tasks[tasks[:, 13] != 0]
        assert plan.learned_matrices == 2 and len(learned) == 5 + 16
        assert set(learned[:, 28].tolist()) == ({5 + 16} if moves else {0})
        filters = [p for p in sim._plans if p.name == "hip_linearfilter"]
        assert bool(filters) != moves
        if filters:
            order = list(sim._plans)
            assert order.index(filters[0]) > order.index(plan)


# more groups than run at once: the last ones read long after the first rule's are through
@pytest.mark.gpu
@pytest.mark.parametrize("shared", [s for s, _ in SHARED])
def test_rules_that_share_activities(queue, shared):
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    rows = 1000 if shared == "rows" else 12000
    (model, probes), (model_o, probes_o) = (rules_on_one_activity(rows, shared) for _ in range(2))
    with Simulator(None, model=model, seed=1) as gpu, OracleSimulator(None, model=model_o, seed=1) as cpu:
        assert any(getattr(p, "learned_matrices", 0) == 2 for p in gpu._plans)
        for steps in (1, 20):
            gpu.run_steps(steps)
            cpu.run_steps(steps)
            for key in probes:
                assert np.array_equal(gpu.data[probes[key]], cpu.data[probes_o[key]])
            assert_same_signals(gpu, cpu)


@pytest.mark.parametrize("dims,columns", [(1, 0), (4, 0), (5, 3), (8, 3)])
def test_few_rows_are_read_whole(monkeypatch, dims, columns):
    """... in the groups of learned rows, each of them once."""
    from nengo_ocl_amd import configs
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    net = configs.c4_pes(1, n_triples=3, n_neurons=1024, dims=dims)[0]
    with Simulator(net, seed=1, event_calibration_steps=0) as sim:
        plan, = [p for p in sim._plans if getattr(p, "learned_matrices", 0)]
        name, args = plan.laid_out[0].__name__ if plan.laid_out else plan.kern.__name__, (plan.laid_out or (0, plan.args))[1]
        assert name == ("nhip_gemv_learn_events" if columns else "nhip_gemv_learn")
        # (the others that are applied to spikes: of the errors' inputs and the probes, see `configs.c4_pes`)
        assert (args[12] if columns else 0) >= columns
        if not columns:
            covered = [y + (r + k) * s for y, s, r, c in plan.host_learn[0][:, [4, 5, 11, 12]].tolist() for k in range(c)]
            assert sorted(covered) == sorted(
                g["y_start"] + r * g["y_stride0"] for g in (plan.prog.geometry[b] for b in plan.members)
                for r in range(g["y_len"]))


def test_launches_that_list_columns_are_looked_at_by_the_calibration(monkeypatch):
    """... and products of populations that spike densely are not among these columns."""
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    for n in (1050, 2048):  # (either way into the launch)
        model = network(n, 32)[0].build_model(dt=0.001)
        with Simulator(None, model=model, seed=1) as sim:
            assert learning_launch(sim).event_driven and sim.event_calibration is not None
            sources = sim._event_spike_sources
        with Simulator(None, model=model, seed=1, _spike_sources_read_whole=sources) as sim:
            assert not any(getattr(p, "event_driven", False) for p in sim._plans)
            assert not any(p.laid_out[1][12] for p in sim._plans if getattr(p, "laid_out", None) is not None
                           and p.laid_out[0].__name__ == "nhip_gemv_learn_events")


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1050, 2048])
def test_populations_that_spike_densely_beside_learned_rows(queue, n):
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    (net, probes), (net_o, probes_o) = (network(n, 32) for _ in range(2))
    with Simulator(net, dt=0.008, seed=1) as gpu, OracleSimulator(net_o, dt=0.008, seed=1) as cpu:
        assert gpu.event_calibration["populations_switched_to_dense_products"] > 0, gpu.event_calibration
        for steps in (1, 20):
            gpu.run_steps(steps)
            cpu.run_steps(steps)
            for p, p_o in zip(probes, probes_o):
                assert np.array_equal(gpu.data[p], cpu.data[p_o])
            assert_same_signals(gpu, cpu)


# two and three filters of the rules and others of any length: all threads, waves with one to four each, two rounds of them
@pytest.mark.gpu
@pytest.mark.parametrize("rule", ["Oja", "BCM"])
@pytest.mark.parametrize("sizes", [[], [1], [3, 70], [5, 64, 257, 30], [1030] + [2, 33, 257, 7] * 2, [9, 260, 2100, 61] * 5])
def test_filters_behind_the_last_reader(queue, rule, sizes):
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    def make():
        rng = np.random.RandomState(3)
        net = mb.Network(seed=5, solver="surrogate")
        stim = net.Node(mb.WhiteSignal(period=0.5, high=6.0, seed=3), size_out=2)
        pre, post = net.Ensemble(130, 2), net.Ensemble(101, 2)
        net.Connection(stim, pre, synapse=None)
        learning = mb.Oja(learning_rate=1e-6, beta=0.7) if rule == "Oja" else mb.BCM(learning_rate=1e-9)
        net.Connection(pre.neurons, post.neurons, transform=rng.normal(scale=1e-3, size=(101, 130)),
                       learning_rule=learning, synapse=mb.Lowpass(0.005))
        probes = [net.Probe(post.neurons, sample_every=0.005)]
        for k, n in enumerate(sizes):
            ens = net.Ensemble(n, 2)
            net.Connection(stim, ens, synapse=None)
            probes.append(net.Probe(ens.neurons, synapse=mb.Lowpass(0.002 + 0.001 * k), sample_every=0.005))
        return net, probes

    (net, probes), (net_o, probes_o) = make(), make()
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        plan, = [p for p in gpu._plans if getattr(p, "learned_matrices", 0)]
        assert plan.args[9] == (2 if rule == "Oja" else 3) + len(sizes)
        for steps in (1, 30):
            gpu.run_steps(steps)
            cpu.run_steps(steps)
            for p, p_o in zip(probes, probes_o):
                assert np.array_equal(gpu.data[p], cpu.data[p_o])
            assert_same_signals(gpu, cpu)
