"""Products with constant matrices on copies of them (csrc/gemv_dots.hip), at the sizes where rows, tiles, passes and
groups have edges, against the CPU oracle bit for bit (they keep the reference's order of summation, so the tolerance
is zero)."""

import numpy as np
import pytest

from helpers import assert_same_signals, host_simulators


def network(n, m, neuron="LIFRate", odd=False, synapses=2, items=2):
    """Populations of `n` neurons whose activities are multiplied by `m` x `n` matrices, with filters of first and
    second order behind them."""
    from nengo_ocl_amd import minibuilder as mb

    rng = np.random.RandomState(n + m)
    net = mb.Network(seed=4, solver="surrogate")
    stim = net.Node(mb.WhiteSignal(period=0.3, high=8.0, seed=4), size_out=2)
    outs = []
    for k in range(items):
        ens = net.Ensemble(n, 2, neuron_type=getattr(mb, neuron)())
        net.Connection(stim, ens, synapse=mb.Lowpass(0.005))
        weights = rng.normal(size=(m + k, n)) / n
        if odd:  # (0 * inf is not a number, wherever the neuron is silent)
            weights[0, -1], weights[-1, n // 2] = np.inf, np.nan
        for s in range(synapses):
            out = net.Node(None, size_in=m + k)
            net.Connection(ens.neurons, out, transform=weights, synapse=[mb.Lowpass(0.005), mb.Alpha(0.01)][s])
            outs.append(net.Probe(out))
    return net, outs


def laid_out(sim):
    return [p for p in sim._plans if getattr(p, "laid_out", None) is not None and hasattr(p, "host_records")]


# one to eight quads of a tile, two tiles, rows that share a record: 4, 8 and 16 tiles and one column more, two passes
# (of more rows than take a group each); groups that end inside their rows
SIZES = [(2, 2), (3, 70), (16, 5), (17, 2), (33, 9), (100, 1), (127, 3), (128, 40), (129, 3), (200, 17), (256, 30),
         (257, 3), (511, 17), (512, 16), (513, 7), (1000, 9), (1024, 8), (1025, 3), (1500, 50), (2048, 5), (2050, 600)]


@pytest.mark.gpu
@pytest.mark.parametrize("neuron", ["LIFRate", "LIF"])
@pytest.mark.parametrize("n,m", SIZES)
def test_rows_of_constant_matrices(queue, monkeypatch, n, m, neuron):
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    (net, probes), (net_o, probes_o) = (network(n, m, neuron) for _ in range(2))
    with Simulator(net, seed=1, event_calibration_steps=0) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        assert laid_out(gpu), [str(p) for p in gpu._plans]
        for steps in (1, 25):
            gpu.run_steps(steps)
            cpu.run_steps(steps)
            for p, p_o in zip(probes, probes_o):
                assert np.array_equal(gpu.data[p], cpu.data[p_o])
            assert_same_signals(gpu, cpu)


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(30, 3), (100, 5), (300, 20), (1001, 20)])
def test_rows_with_values_that_are_not_finite(queue, monkeypatch, n, m):
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    (net, _), (net_o, _) = (network(n, m, odd=True) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        assert laid_out(gpu)
        gpu.run_steps(20)
        cpu.run_steps(20)
        assert_same_signals(gpu, cpu)


@pytest.mark.gpu
def test_matrices_that_the_host_changes(queue, monkeypatch):
    from nengo_ocl_amd.simulator import Simulator
    from oracle.oracle_sim import OracleSimulator

    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    (net, _), (net_o, _) = (network(300, 20, synapses=1) for _ in range(2))
    with Simulator(net, seed=1) as gpu, OracleSimulator(net_o, seed=1) as cpu:
        for sim, of in ((gpu, net), (cpu, net_o)):
            sim.run_steps(5)
            sig, = {op.A.base for op in sim.model.operators if getattr(op, "A", None) is not None
                    and op.A.base.shape == (20, 300)}
            sim.signals[sig] = 2.5 * sim.signals[sig][::-1]
            sim.run_steps(5)
        assert_same_signals(gpu, cpu)


@pytest.mark.parametrize("n,m", SIZES)
def test_records_cover_every_row_once(monkeypatch, n, m):
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    with Simulator(network(n, m)[0], seed=1, event_calibration_steps=0) as sim:
        plans = [p for p in laid_out(sim) if any(
            p.prog.geometry[b]["dots"][0]["a_shape1"] == n for b in p.members)]
        assert plans
        for plan in plans:
            tiles, quads, _, _, n_groups = plan.laid_out[1][:5]
            records, geometry = plan.host_records, plan.prog.geometry
            rows = sorted(g["y_start"] + r * g["y_stride0"] for g in (geometry[b] for b in plan.members)
                          for r in range(g["y_len"]))
            if tiles <= 2:
                assert len(records) == n_groups * 64 // tiles
                real = records[records[:, 3] >= 0]
                assert sorted(real[:, 4].tolist()) == rows and len(records) - len(real) < 64 // tiles
                assert max(real[:, 2]) <= 128 * tiles and max(min(c, 128) for c in real[:, 2]) <= 16 * quads
            else:
                assert len(records) == n_groups and records[:, 6].max() <= 64 // tiles
                assert sorted(y + (r + k) * stride for y, stride, r, count in records[:, [8, 9, 5, 6]].tolist()
                              for k in range(count)) == rows


def test_chains_divided_over_launches(monkeypatch):
    """What a chain of short operations begins with rides in the launch before the one that carries the rest."""
    from nengo_ocl_amd import configs
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    net = configs.c2_watts_strogatz(1, n_ens=64, n_neurons=100, n_driven=2)[0]
    with Simulator(net, seed=1, event_calibration_steps=0) as sim:
        runs = [[p.name for p in q.runs.members] for q in sim._plans if getattr(q, "runs", None) is not None]
        assert len(runs) == 2 and runs[0] == ["hip_timeupdate", "hip_presentinput"], runs
        assert "hip_linearfilter" in runs[1]
        whole, = [q.carried for q in sim._plans if getattr(q, "carried", None) is not None]
        assert sorted(runs[0] + runs[1]) == sorted(p.name for p in whole.members)


def test_launches_of_more_than_the_memory_side_cache_holds_read_matrices_as_they_lie(monkeypatch):
    from nengo_ocl_amd import hipra_dots
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    for limit, expected in ((1 << 30, True), (100 * 16 * 40 * 4, False)):
        monkeypatch.setattr(hipra_dots, "MAX_BYTES", limit)
        with Simulator(network(1500, 50)[0], seed=1) as sim:
            assert bool(laid_out(sim)) == expected


# rows x columns (x items) of a launch: lane or four lanes per row, streamed on 16-byte boundaries and not, any shape;
# what its widest matrix makes of the others; on both sides of each limit
@pytest.mark.parametrize("shapes,expected", [
    ([(50, 2, 20)], True), ([(105000, 2, 1)], True), ([(115000, 2, 1)], False), ([(2000, 4, 60)], False),
    ([(50, 5, 3000)], True), ([(100, 2, 10), (10, 30, 1)], True), ([(100, 2, 10), (10, 100, 1)], False),
    ([(100, 2, 10), (10, 250, 1)], True), ([(500, 2, 50), (10, 250, 1)], False), ([(170000, 8, 1)], True),
    ([(180000, 8, 1)], False), ([(180000, 32, 1)], False), ([(180000, 15, 1)], False), ([(180000, 31, 1)], True),
    ([(180000, 40, 1)], True), ([(300000, 40, 1)], False), ([(120000, 68, 1)], False), ([(150000, 100, 1)], True),
    ([(60000, 132, 1)], False), ([(110000, 66, 1)], True), ([(9000, 520, 1)], True)])
def test_copies_that_read_much_more_than_their_matrices_are_not_made(monkeypatch, shapes, expected):
    check_layout(monkeypatch, shapes, expected, 0.005)


@pytest.mark.parametrize("shapes,expected", [
    ([(50000, 128, 1)], True), ([(64000, 128, 1)], False), ([(2000, 51, 40)], True), ([(2000, 51, 60)], False),
    ([(27000, 200, 1)], True), ([(40000, 200, 1)], False), ([(2000, 66, 40)], True), ([(64, 4096, 40)], True)])
def test_large_copies_are_not_made_for_launches_without_filters(monkeypatch, shapes, expected):
    check_layout(monkeypatch, shapes, expected, None)


def check_layout(monkeypatch, shapes, expected, synapse):
    from nengo_ocl_amd import minibuilder as mb
    from nengo_ocl_amd.simulator import Simulator

    host_simulators(monkeypatch)
    monkeypatch.setenv("NENGO_HIP_RESIDENT", "0")
    net = mb.Network(seed=4, solver="surrogate")
    stim = net.Node(mb.WhiteSignal(period=0.3, high=8.0, seed=4), size_out=1)
    for m, n, items in shapes:
        for k in range(items):
            ens, out = net.Ensemble(n, 1, neuron_type=mb.LIFRate()), net.Node(None, size_in=m)
            net.Connection(stim, ens, synapse=None)
            weights = np.broadcast_to(np.float64(k + 1.0), (m, n))
            net.Connection(ens.neurons, out, transform=weights, synapse=synapse)
            net.Probe(out[:1], synapse=0.01)
    with Simulator(net, seed=1) as sim:
        plan, = [p for p in sim._plans if hasattr(p, "prog") and any(
            d["a_shape1"] == shapes[0][1] and p.prog.geometry[b]["y_len"] == shapes[0][0]
            for b in p.members for d in p.prog.geometry[b]["dots"])]
        assert (plan in laid_out(sim)) == expected, (plan.kernel_class, str(plan))
