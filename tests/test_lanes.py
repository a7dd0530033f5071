"""Launches that update neurons with a lane per neuron (csrc/gemv_lanes.hip), at the sizes where their tasks, column
quads and passes have edges, against the CPU oracle bit for bit (they keep the reference's order of summation, so the
tolerance is zero)."""

import numpy as np
import pytest

from helpers import assert_same_signals, host_simulators


def network(n, d, neuron, seed=3):
    """Populations whose input is a sum of up to nine parts, of one part, a node's value, and nothing."""
    from nengo_ocl_amd import minibuilder as mb

    net = mb.Network(seed=seed, solver="surrogate")
    make = lambda n: net.Ensemble(n, d, neuron_type=neuron())
    ens = [make(n), make(n + 1), make(max(n - 1, 1)), make(n)]
    stim = net.Node(mb.WhiteSignal(period=0.3, high=8.0, seed=4), size_out=d)
    net.Connection(stim, ens[0], synapse=mb.Lowpass(0.005))
    for k in range(8):
        net.Connection(ens[k % 2], ens[0], transform=0.1 + 0.05 * k, synapse=mb.Lowpass(0.002 + 0.001 * k))
    net.Connection(ens[0], ens[1], synapse=mb.Alpha(0.01))
    net.Connection(stim, ens[2], synapse=None)
    return net, [net.Probe(e, synapse=0.01) for e in ens] + [net.Probe(ens[1].neurons)]


def laid_out(sim):
    return [p for p in sim._plans if getattr(p, "laid_out", None) is not None and hasattr(p, "host_pops")]


@pytest.mark.gpu
@pytest.mark.parametrize("neuron", ["LIF", "AdaptiveLIF", "LIFRate", "RectifiedLinear", "SpikingRectifiedLinear"])
# one to four columns are read as they lie; quads of one, two and three columns; 16 quads and one more, 32; tasks of
# 63, 64 and 65 rows; items of the small and of the large kernel, on 16-byte boundaries and not
@pytest.mark.parametrize("n,d", [(2, 1), (63, 2), (64, 3), (65, 4), (200, 5), (70, 7), (129, 8), (301, 30), (601, 18),
                                 (200, 50), (140, 62), (300, 63), (129, 64), (260, 65), (100, 100), (300, 127),
                                 (65, 128)])
def test_neurons_a_lane_each(queue, monkeypatch, neuron, n, d):
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    (net, probes), (net_o, probes_o) = (network(n, d, getattr(mb, neuron)) for _ in range(2))
    with Simulator(net, seed=1, event_calibration_steps=0) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        assert laid_out(gpu), [str(p) for p in gpu._plans]
        for steps in (1, 30):
            gpu.run_steps(steps)
            cpu.run_steps(steps)
            for p, p_o in zip(probes, probes_o):
                assert np.array_equal(gpu.data[p], cpu.data[p_o])
            assert_same_signals(gpu, cpu)


@pytest.mark.gpu
def test_encoders_that_the_host_changes(queue, monkeypatch):
    """A write reaches the copy that the launch reads, a reset takes it back."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    (net, _), (net_o, _) = (network(200, 50, mb.LIF) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        for change in (False, True):
            for sim, ens in ((gpu, net.ensembles[0]), (cpu, net_o.ensembles[0])):
                if change:
                    sig = sim.model.sig[ens]["encoders"]
                    sim.signals[sig] = 1.5 * sim.signals[sig][::-1]
                sim.run_steps(10)
            assert_same_signals(gpu, cpu)
        gpu.reset()
        with OracleSimulator(network(200, 50, mb.LIF)[0], seed=1) as fresh:
            for sim in (gpu, fresh):
                sim.run_steps(10)
            assert_same_signals(gpu, fresh)


@pytest.mark.parametrize("n,d", [(2, 1), (64, 3), (65, 4), (301, 30), (200, 50), (300, 127)])
def test_tasks_cover_every_neuron_once(monkeypatch, n, d):
    """Records of at most 64 rows from multiples of 64 on, matrices apart in the copy, groups of four filled
    up with tasks of no rows."""
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    with Simulator(network(n, d, mb.LIF)[0], seed=1, event_calibration_steps=0) as sim:
        assert laid_out(sim)
        for plan in laid_out(sim):
            tasks, geometry = plan.host_tasks, plan.prog.geometry
            assert plan.laid_out[1][2] % 4 == 0 and plan.laid_out[1][2] - len(tasks) < 4
            blocks = []
            for b in plan.members:
                mine = tasks[tasks[:, 0] == b]
                mine = mine[np.argsort(mine[:, 1])]
                assert not np.any(mine[:, 1] % 64) and mine[:, 2].max() <= 64
                assert np.array_equal(np.concatenate([r + np.arange(m) for r, m in mine[:, 1:3]]),
                                      np.arange(geometry[b]["y_len"]))
                for dot in geometry[b]["dots"][:1]:
                    if d > 4:
                        quads = -(-dot["a_shape1"] // 4)
                        assert set(mine[:, 17]) == {quads} and len(set(mine[:, 16])) == 1
                        blocks.append((int(mine[0, 16]), -(-geometry[b]["y_len"] // 64) * quads))
                    else:
                        assert set(mine[:, 16]) == {dot["a_start"]} and np.all(mine[:, 21] < 0)
            blocks = sorted(set(blocks))
            assert all(a + size <= b for (a, size), (b, _) in zip(blocks, blocks[1:]))


@pytest.mark.parametrize("groups", [1, 7, 8, 9, 63, 64, 1000])
def test_groups_of_a_die_are_neighbours_in_the_list(groups):
    from nengo_ocl_amd import hipra_lanes

    tasks = np.arange(1, 4 * groups)[:, None] * np.ones((1, 3), dtype=np.int32)
    out = hipra_lanes.for_the_dies(tasks.astype(np.int32))[:, 0].reshape(groups, 4)
    assert sorted(out.ravel()) == [0] + list(range(1, 4 * groups))
    for die in range(8):
        firsts = out[die::8, 0]
        assert np.all(np.diff(firsts) == 4)


def populations(n, dims, neuron="LIF", idle=True):
    """Populations that send decoded vectors to each other and to a node of nobody's, one (`idle`) without input."""
    from nengo_ocl_amd import minibuilder as mb

    net = mb.Network(seed=4, solver="surrogate")
    stim = net.Node(mb.WhiteSignal(period=0.3, high=8.0, seed=4), size_out=dims)
    ens = [net.Ensemble(n + k, dims, neuron_type=getattr(mb, neuron)()) for k in range(4)]
    for k, post in enumerate(ens[:3] if idle else ens):
        net.Connection(stim, post, synapse=mb.Lowpass(0.005))
        for pre in (ens[3], ens[(k + 1) % 3], ens[(k + 2) % 3]):
            net.Connection(pre, post, transform=0.3, synapse=mb.Lowpass(0.005))
    spare = net.Node(None, size_in=dims)
    for pre in ens[:2]:
        net.Connection(pre, spare, synapse=mb.Lowpass(0.005))
    return net, [net.Probe(ens[0], synapse=0.01), net.Probe(spare), net.Probe(ens[3], synapse=0.01)]


# four lanes or one per row of small matrices, large ones of any shape, of quads and back to back; sums of up to 64
# elements and of more, part of them in a node's place
POPULATIONS = [(60, 1), (150, 4), (90, 7), (250, 37), (220, 64), (210, 65), (214, 86), (130, 128), (900, 94), (700, 3)]


@pytest.mark.gpu
@pytest.mark.parametrize("neuron", ["LIF", "Sigmoid"])
@pytest.mark.parametrize("idle", [False, True])
@pytest.mark.parametrize("n,dims", POPULATIONS)
def test_input_sums_and_populations_without_input(queue, monkeypatch, n, dims, idle, neuron):
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    (net, probes), (net_o, probes_o) = (populations(n, dims, neuron, idle) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        names = [p.laid_out[0].__name__ if p.laid_out else p.kern.__name__ for p in gpu._plans
                 if getattr(p, "kern", None)]
        assert "nhip_gemv_lanes" in names and "nhip_gemv" not in names and len(names) <= 3, names
        for steps in (1, 25):
            gpu.run_steps(steps)
            cpu.run_steps(steps)
            for p, p_o in zip(probes, probes_o):
                assert np.array_equal(gpu.data[p], cpu.data[p_o])
            assert_same_signals(gpu, cpu)


@pytest.mark.parametrize("n,dims", POPULATIONS)
def test_input_sums_are_formed_once(monkeypatch, n, dims):
    """Every sum belongs to a record of the neurons' launch, also one that no population reads."""
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    with Simulator(populations(n, dims)[0], seed=1) as sim:
        plan, = [p for p in sim._plans if p.laid_out and p.laid_out[0].__name__ == "nhip_gemv_lanes"]
        tasks = plan.host_tasks
        parts = tasks[(tasks[:, 11] > 0) & (tasks[:, 1] == 0)][:, 11]
        assert sorted(parts.tolist()) == [1, 1, 2, 4, 4, 4]  # (two of probes)
        assert sorted(set(tasks[tasks[:, 9] == 0][:, 11].tolist())) == [0, 1, 2]


def many_matrices(neuron):
    """Encoders and decoders of seven populations of one launch each."""
    from nengo_ocl_amd import minibuilder as mb

    net = mb.Network(seed=2, solver="surrogate")
    stim = net.Node(mb.WhiteSignal(period=0.3, high=8.0, seed=4), size_out=6)
    probes = []
    for k in range(7):
        ens = net.Ensemble(70 + k, 6, neuron_type=neuron())
        net.Connection(stim, ens, synapse=mb.Lowpass(0.005))
        probes.append(net.Probe(ens, synapse=0.01))
    return net, probes


@pytest.mark.parametrize("limit", [1, 3, 7])
def test_matrices_are_laid_out_in_launches_that_hold_them(monkeypatch, limit):
    from nengo_ocl_amd import hipra_gemv, hipraggedarray, minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    monkeypatch.setattr(hipra_gemv, "LAY_OUT_MATRICES", limit)
    calls, make = {}, hipraggedarray.Queue

    def queue(device=0):
        q = make(device)

        class Lib:
            def __getattr__(self, name, lib=q.lib):
                entry = getattr(lib, name)
                if name not in ("nhip_lay_out_lanes", "nhip_lay_out_dots"):
                    return entry

                def lay_out(handle, matrices, n, *rest):
                    calls.setdefault(name, []).append((matrices.value, n))
                    return -1 if n > limit else 0

                return lay_out

        q.lib = Lib()
        return q

    monkeypatch.setattr(hipraggedarray, "Queue", queue)
    with Simulator(many_matrices(mb.LIFRate)[0], seed=1):
        assert set(calls) == {"nhip_lay_out_lanes", "nhip_lay_out_dots"}
        for made in calls.values():
            assert sum(n for _, n in made) == 7 and [at - made[0][0] for at, _ in made] == [
                32 * limit * k for k in range(-(-7 // limit))]


@pytest.mark.gpu
def test_matrices_that_several_launches_lay_out(queue, monkeypatch):
    from nengo_ocl_amd import hipra_gemv, minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    monkeypatch.setattr(hipra_gemv, "LAY_OUT_MATRICES", 3)
    (net, probes), (net_o, probes_o) = (many_matrices(mb.LIFRate) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        assert len([p for p in gpu._plans if p.laid_out is not None]) == 2
        gpu.run_steps(20)
        cpu.run_steps(20)
        for p, p_o in zip(probes, probes_o):
            assert np.array_equal(gpu.data[p], cpu.data[p_o])
        assert_same_signals(gpu, cpu)


@pytest.mark.parametrize("limit,past", [(330e6, False), (1e3, True)])
def test_steps_that_move_more_than_the_cache_keeps_read_past_it(monkeypatch, limit, past):
    """... all that moves in the step counts, of launches that visit active columns only a part."""
    from nengo_ocl_amd import configs, hipra_lanes, minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setattr(hipra_lanes, "STEP_BYTES", limit)
    for net in (network(300, 30, mb.LIF)[0], configs.c3_large(n_ens=3, n_neurons=1024, dims=16, fan_out=2)[0]):
        with Simulator(net, seed=1, event_calibration_steps=0) as sim:
            kinds = [p.laid_out[1][0] for p in laid_out(sim)]
            assert kinds and all(k == (1 | 16 if past else 1) for k in kinds)
            moved = sum((p.bw_per_call or 0) * (0.1 if getattr(p, "event_driven", False) else 1) for p in sim._plans)
        for share, expected in ((0.5, True), (2.0, False)):
            monkeypatch.setattr(hipra_lanes, "STEP_BYTES", share * moved)
            with Simulator(net, seed=1, event_calibration_steps=0) as sim:
                assert all(bool(p.laid_out[1][0] & 16) == expected for p in laid_out(sim))
        monkeypatch.setattr(hipra_lanes, "STEP_BYTES", limit)


def test_matrices_read_past_the_cache_do_not_count(monkeypatch):
    """Decoders of rate neurons that keep the launch with non-temporal loads."""
    from nengo_ocl_amd import hipra_dots, hipra_lanes, minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setattr(hipra_dots, "MAX_BYTES", 0)
    net = mb.Network(seed=2, solver="surrogate")
    ens = [net.Ensemble(1024, 64, neuron_type=mb.LIFRate()) for _ in range(40)]
    for a, b in zip(ens, ens[1:] + ens[:1]):
        net.Connection(a, b, synapse=mb.Lowpass(0.005))
    with Simulator(net, seed=1) as sim:
        own = sum(p.bw_per_call for p in laid_out(sim))
        others = sum(p.bw_per_call for p in sim._plans if p.name == "hipra_gemv.tile_filter" and p.laid_out is None)
    assert others > 0.5 * own > 0
    for limit, expected in ((1.4 * own, False), (0.9 * own, True)):
        monkeypatch.setattr(hipra_lanes, "STEP_BYTES", limit)
        with Simulator(net, seed=1) as sim:
            assert all(bool(p.laid_out[1][0] & 16) == expected for p in laid_out(sim))


@pytest.mark.gpu
@pytest.mark.parametrize("neuron", ["LIF", "LIFRate"])
@pytest.mark.parametrize("n,d", [(65, 4), (200, 5), (129, 8), (301, 30), (129, 64), (260, 65), (65, 128)])
def test_neurons_whose_encoders_are_read_past_the_cache(queue, monkeypatch, neuron, n, d):
    from nengo_ocl_amd import hipra_lanes, minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    monkeypatch.setattr(hipra_lanes, "STEP_BYTES", 0)
    (net, probes), (net_o, probes_o) = (network(n, d, getattr(mb, neuron)) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        assert laid_out(gpu) and all(p.laid_out[1][0] & 16 for p in laid_out(gpu))
        gpu.run_steps(25)
        cpu.run_steps(25)
        for p, p_o in zip(probes, probes_o):
            assert np.array_equal(gpu.data[p], cpu.data[p_o])
        assert_same_signals(gpu, cpu)


@pytest.mark.parametrize("several,others,expected", [(1, 4, True), (2, 2, True), (3, 2, False), (4, 0, False)])
def test_small_items_with_several_products_keep_their_launch(monkeypatch, several, others, expected):
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    net = mb.Network(seed=1, solver="surrogate")
    stim = net.Node(mb.WhiteSignal(period=0.3, high=8.0, seed=4), size_out=2)
    sources = [net.Ensemble(3, 1, neuron_type=mb.LIFRate()) for _ in range(3)]
    for k in range(several + others):
        ens = net.Ensemble(200 + k, 2)
        net.Connection(stim, ens, synapse=mb.Lowpass(0.005))
        for source in sources if k < several else ():
            net.Connection(source.neurons, ens.neurons, transform=np.full((200 + k, 3), 1e-3), synapse=None)
    with Simulator(net, seed=1, event_calibration_steps=0) as sim:
        plan, = [p for p in sim._plans if getattr(p, "name", "") == "hipra_gemv.wave_ref_lif"
                 and any(p.prog.geometry[b]["y_len"] >= 200 for b in p.members)]
        counts = [len(plan.prog.geometry[b]["dots"]) for b in plan.members]
        assert sum(c > 1 for c in counts) == several
        assert (plan.laid_out is not None) == expected
