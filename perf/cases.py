"""What the framework is timed on: whole simulations, run the way a user's program runs them.

A case is a network, a number of timesteps per call and the neuron type and synapse options
in use.  `prepare` builds the network (seeded) and its `Simulator`; `run` advances it by one
call and takes what the program asked for: the probe samples of that call and, where the
network learns, the learned matrices.

Kinds of network (sizes of the listed cases are those of `nengo_ocl_amd.configs`, the tests
and the benchmark, or generic; `draw` spreads them):

* ``readme``     two small scalar populations: what a first program does; a closed loop asks
                 for one step per call, an experiment for a second of simulated time
* ``circconv``   circular convolution: an array of small product ensembles between dense
                 transforms
* ``smallworld`` many small ensembles, every edge a decoded connection
* ``ensembles``  few to many large ensembles that send decoded vectors to each other:
                 spiking or rate neurons, first- or second-order synapses, any dimension
* ``pes``        decoders learned from an error signal
* ``hebbian``    weights between two neuron populations learned by Oja's or the BCM rule
* ``sparse``     one population with a sparse recurrent weight matrix
* ``vision``     an image through two convolution layers of neurons into a readout
"""

import numpy as np

from nengo_ocl_amd import Simulator, configs
from nengo_ocl_amd import minibuilder as mb

NEURONS = {"LIF": mb.LIF, "LIFRate": mb.LIFRate, "AdaptiveLIF": mb.AdaptiveLIF,
           "RectifiedLinear": mb.RectifiedLinear, "Sigmoid": mb.Sigmoid,
           "SpikingRectifiedLinear": mb.SpikingRectifiedLinear}
SPIKING = ("LIF", "AdaptiveLIF", "SpikingRectifiedLinear")
# neurons of the spiking types fire in 8 % of the steps on average (rates of 200-400 Hz at
# full drive): only those columns of a matrix applied to spikes cannot be done without
SPIKE_SHARE = 0.08


def listed():
    return [
        # a closed loop (robot, interactive session): one step per call, latency is all
        {"name": "readme_one_step", "kind": "readme", "neurons": 100, "steps": 1},
        # the first program of the documentation: one simulated second
        {"name": "readme_second", "kind": "readme", "neurons": 100, "steps": 1000},
        # binding of two semantic pointers
        {"name": "circconv_64", "kind": "circconv", "dims": 64, "steps": 200},
        # a network of many scalar populations
        {"name": "smallworld_256", "kind": "smallworld", "ensembles": 256, "neurons": 100,
         "steps": 200},
        # the bandwidth-bound network of the benchmark: a million neurons
        {"name": "ensembles_256x4096x64", "kind": "ensembles", "ensembles": 256, "neurons": 4096,
         "dims": 64, "neuron": "LIF", "synapse": "lowpass", "steps": 100},
        # a mid-sized model with sizes nobody rounded
        {"name": "ensembles_37x1501x50", "kind": "ensembles", "ensembles": 37, "neurons": 1501,
         "dims": 50, "neuron": "LIF", "synapse": "lowpass", "steps": 100},
        # the same kind of model tuned with rate neurons, second-order synapses
        {"name": "rate_48x2000x32", "kind": "ensembles", "ensembles": 48, "neurons": 2000,
         "dims": 32, "neuron": "LIFRate", "synapse": "alpha", "steps": 100},
        # adaptive neurons in a cortical-style model
        {"name": "adaptive_32x1000x16", "kind": "ensembles", "ensembles": 32, "neurons": 1000,
         "dims": 16, "neuron": "AdaptiveLIF", "synapse": "lowpass", "steps": 100},
        # supervised learning: 64 decoders learned at once, fetched after the call
        {"name": "pes_64x2000x32", "kind": "pes", "ensembles": 64, "neurons": 2000, "dims": 32,
         "steps": 500},
        # unsupervised learning between two layers of neurons
        {"name": "oja_2000", "kind": "hebbian", "neurons": 2000, "rule": "Oja", "steps": 200},
        # the sparse recurrent population of the benchmark script
        {"name": "sparse_100k", "kind": "sparse", "neurons": 100000, "fan_out": 100, "steps": 100},
        # an image classifier's first layers
        {"name": "vision_28", "kind": "vision", "size": 28, "channels": 1, "filters": 32,
         "neuron": "RectifiedLinear", "steps": 50},
    ]


def _log_int(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["readme", "circconv", "smallworld", "ensembles", "ensembles", "pes",
                       "hebbian", "sparse", "vision"])
    if kind == "readme":
        return {"kind": kind, "neurons": _log_int(rng, 30, 1000),
                "steps": rng.choice([1, _log_int(rng, 2, 1500)])}
    if kind == "circconv":
        return {"kind": kind, "dims": _log_int(rng, 8, 128), "steps": _log_int(rng, 10, 300)}
    if kind == "smallworld":
        return {"kind": kind, "ensembles": _log_int(rng, 16, 300), "neurons": _log_int(rng, 20, 150),
                "steps": _log_int(rng, 10, 300)}
    if kind == "ensembles":
        dims, neurons = _log_int(rng, 2, 100), _log_int(rng, 200, 5000)
        ensembles = max(2, min(_log_int(rng, 4, 200), 12000000 // (dims * neurons)))
        return {"kind": kind, "ensembles": ensembles, "neurons": neurons, "dims": dims,
                "neuron": rng.choice(sorted(NEURONS) + ["LIF", "LIF"]),
                "synapse": rng.choice(["lowpass", "lowpass", "alpha"]),
                "steps": _log_int(rng, 20, 100)}
    if kind == "pes":
        dims, neurons = _log_int(rng, 2, 64), _log_int(rng, 100, 3000)
        ensembles = max(1, min(_log_int(rng, 1, 60), 3000000 // (dims * neurons)))
        return {"kind": kind, "ensembles": ensembles, "neurons": neurons, "dims": dims,
                "steps": _log_int(rng, 100, 500)}
    if kind == "hebbian":
        return {"kind": kind, "neurons": _log_int(rng, 50, 2500), "rule": rng.choice(["Oja", "BCM"]),
                "steps": _log_int(rng, 20, 300)}
    if kind == "sparse":
        return {"kind": kind, "neurons": _log_int(rng, 2000, 100000), "fan_out": _log_int(rng, 5, 100),
                "steps": _log_int(rng, 20, 200)}
    return {"kind": kind, "size": rng.randint(12, 48), "channels": rng.choice([1, 3]),
            "filters": rng.randint(4, 40), "neuron": rng.choice(["RectifiedLinear", "LIF"]),
            "steps": _log_int(rng, 10, 100)}


def _synapse(case):
    return mb.Alpha(0.01) if case["synapse"] == "alpha" else mb.Lowpass(0.005)


def _ensembles(case, seed):
    """Every ensemble sends its decoded vector to up to four others (`configs.c3_large`)."""
    n_ens, n, d = case["ensembles"], case["neurons"], case["dims"]
    rng = np.random.RandomState(seed)
    net = mb.Network(seed=seed, share_decoded=True, solver="surrogate")
    # encoders: unit vectors; windows of one pool, since drawing them costs more than using them
    pool = rng.standard_normal((2 * n + 64 * n_ens, d))
    ens = [net.Ensemble(n, d, neuron_type=NEURONS[case["neuron"]](),
                        encoders=pool[int(k):int(k) + n])
           for k in rng.randint(len(pool) - n, size=n_ens)]
    fan_out = min(4, n_ens - 1)
    for i in range(n_ens):
        others = [j for j in range(n_ens) if j != i]
        for j in rng.choice(others, size=fan_out, replace=False):
            net.Connection(ens[i], ens[int(j)], transform=1.0 / fan_out, synapse=_synapse(case))
    drive = net.Node(mb.WhiteSignal(period=1.0, high=5.0, seed=int(rng.randint(2 ** 31 - 1))),
                     size_out=d)
    for k in range(0, n_ens, 8):
        net.Connection(drive, ens[k], synapse=mb.Lowpass(0.005))
    return net, [net.Probe(e, synapse=0.01) for e in ens[:2]]


def _hebbian(case, seed):
    n = case["neurons"]
    rng = np.random.RandomState(seed)
    net = mb.Network(seed=seed, solver="surrogate")
    stim = net.Node(mb.WhiteSignal(period=1.0, high=5.0, seed=int(rng.randint(2 ** 31 - 1))),
                    size_out=2)
    pre, post = net.Ensemble(n, 2), net.Ensemble(n, 2)
    net.Connection(stim, pre, synapse=mb.Lowpass(0.005))
    rule = mb.Oja(learning_rate=1e-6) if case["rule"] == "Oja" else mb.BCM(learning_rate=1e-9)
    net.Connection(pre.neurons, post.neurons, transform=rng.normal(scale=1e-2 / n, size=(n, n)),
                   learning_rule=rule, synapse=mb.Lowpass(0.005))
    return net, [net.Probe(post, synapse=0.01)]


def _vision(case, seed):
    size, channels, filters = case["size"], case["channels"], case["filters"]
    rng = np.random.RandomState(seed)
    net = mb.Network(seed=seed, solver="surrogate")
    kw = dict(neuron_type=NEURONS[case["neuron"]](), max_rates=(100, 200), intercepts=(-0.5, 0.5))
    images = rng.uniform(size=(4, size * size * channels))
    eye = net.Node(mb.PresentInput(images, 0.02), size_out=size * size * channels)
    first = mb.Convolution(filters, (size, size, channels), kernel_size=(3, 3), seed=seed)
    shape = first.spec.output_shape.shape
    second = mb.Convolution(2 * filters, tuple(shape), kernel_size=(3, 3), strides=(2, 2), seed=seed,
                            init=rng.uniform(-1, 1, size=(3, 3, filters, 2 * filters)) / (90.0 * filters))
    one = np.ones((first.size_out, 1))
    layer1 = net.Ensemble(first.size_out, 1, encoders=one, **kw)
    layer2 = net.Ensemble(second.size_out, 1, encoders=np.ones((second.size_out, 1)), **kw)
    net.Connection(eye, layer1.neurons, transform=first, synapse=None)
    net.Connection(layer1.neurons, layer2.neurons, transform=second, synapse=mb.Lowpass(0.005))
    out = net.Node(None, size_in=10)
    net.Connection(layer2.neurons, out, synapse=mb.Lowpass(0.005),
                   transform=rng.normal(scale=1e-2 / second.size_out, size=(10, second.size_out)))
    return net, [net.Probe(out), net.Probe(layer2.neurons, sample_every=0.01)]


def _network(case, seed):
    """(network, probes, connections whose weights are learned)"""
    kind = case["kind"]
    if kind == "readme":
        net, probes, _ = configs.c0_readme(seed, n_neurons=case["neurons"])
        probes = list(probes.values())
    elif kind == "circconv":
        net, probes, _ = configs.c1_circconv(seed, dims=case["dims"])
        net.n_eval_points = 300
        probes = list(probes.values())
    elif kind == "smallworld":
        n = case["ensembles"]
        net, probes, _ = configs.c2_watts_strogatz(seed, n_ens=n, n_neurons=case["neurons"],
                                                   n_driven=max(1, n // 32))
        net.n_eval_points = 300
        probes = list(probes.values())
    elif kind == "ensembles":
        net, probes = _ensembles(case, seed)
    elif kind == "pes":
        net, probes, _ = configs.c4_pes(seed, n_triples=case["ensembles"], n_neurons=case["neurons"],
                                        dims=case["dims"])
        probes = list(probes.values())
    elif kind == "hebbian":
        net, probes = _hebbian(case, seed)
    elif kind == "sparse":
        net, probes, _ = configs.c5_sparse_recurrent(seed, n_neurons=case["neurons"],
                                                     fan_outs=case["fan_out"])
        probes = list(probes.values())
    else:
        net, probes = _vision(case, seed)
    return net, probes, [c for c in net.connections if isinstance(c.learning_rule, (mb.PES, mb.Oja, mb.BCM))]


class _State:
    """A simulator and what its user reads after a call; closed with its last reference."""

    def __init__(self, case, seed):
        # `configs` multiplies the seed by up to 7919, and NumPy takes 32 bits of it
        net, self.probes, learned = _network(case, seed % 500009)
        self.sim = Simulator(net, progress_bar=False)
        self.learned = [self.sim.model.sig[c]["weights"] for c in learned]
        self.steps = case["steps"]
        if case["kind"] == "readme":
            # a loop that is under way: from rest nothing spikes in the first steps
            self.sim.run_steps(250, progress_bar=False)

    def __del__(self):
        if getattr(self, "sim", None) is not None and not self.sim.closed:
            self.sim.close()


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    sim = state.sim
    sim.clear_probes()
    sim.run_steps(state.steps, progress_bar=False)
    out = {"probes": [sim.data[p] for p in state.probes]}
    if state.learned:
        out["learned"] = np.stack([sim.signals[w] for w in state.learned])
    return out


def work(case):
    """Bytes and operations of the steps of one call: every matrix read once per step (of a
    matrix applied to spikes the columns of the neurons that spiked), neuron state, filter
    state and learned matrices read and written once per step."""
    kind, steps = case["kind"], case["steps"]
    share = SPIKE_SHARE if case.get("neuron", "LIF") in SPIKING else 1.0
    words = flops = 0.0
    if kind == "readme":
        n = 2 * case["neurons"]
        words, flops = n * (2 + 4 + 1 + 1), 30.0 * n
    elif kind == "circconv":
        dims = case["dims"]
        products = 4 * (dims // 2 + 1)
        n = 100 * products
        words = 3 * dims * products + n * (2 + 1 + 4 + 1)
        flops = 6.0 * dims * products + 30.0 * n
    elif kind == "smallworld":
        n = case["ensembles"] * case["neurons"]
        edges = min(10, case["ensembles"] - 1) * case["ensembles"]
        words = n * (1 + 1 + 4) + share * edges * case["neurons"] + 4 * edges
        flops = 30.0 * n + 2.0 * share * edges * case["neurons"]
    elif kind == "ensembles":
        n, d = case["ensembles"] * case["neurons"], case["dims"]
        state = {"LIF": 4, "AdaptiveLIF": 6, "SpikingRectifiedLinear": 2}.get(case["neuron"], 0)
        words = n * (d + share * d + 1 + state) + 4 * case["ensembles"] * d
        flops = n * (2.0 * d + 2.0 * share * d + 30)
    elif kind == "pes":
        n, d = case["ensembles"] * case["neurons"], case["dims"]
        # three populations per rule; the learned decoders are read and written, the others
        # applied to spikes
        words = n * (3 * d + 2 * d + 2 * share * d + 3 * 5 + 2)
        flops = n * (6.0 * d + 4.0 * d + 4.0 * share * d + 90)
    elif kind == "hebbian":
        n = case["neurons"]
        words, flops = 2.0 * n * n + 20 * n, (5.0 + 2.0 * share) * n * n
    elif kind == "sparse":
        # value and column index of every stored element
        nnz = case["neurons"] * case["fan_out"]
        words, flops = 2.0 * nnz + 8.0 * case["neurons"], 2.0 * nnz + 30.0 * case["neurons"]
    else:
        size, ch, f = case["size"], case["channels"], case["filters"]
        n1 = (size - 2) ** 2 * f
        n2 = ((size - 5) // 2 + 1) ** 2 * 2 * f
        words = size * size * ch + 9 * ch * f + 18 * f * f + 6.0 * n1 + 16.0 * n2
        flops = 18.0 * ch * n1 + 18.0 * f * n2 + 20.0 * n2 + 10.0 * (n1 + n2)
    return {"bytes": 4.0 * words * steps, "flops": float(flops * steps)}


def tolerance(case):
    # Measured against a NumPy interpretation of the same networks whose products sum in
    # another order: 1e-7 to 2e-7 (largest value 6e-7) as long as no neuron spikes in another
    # step, 6e-4 (5e-3) where one of the 13,200 neurons of circconv_64 does.  Rate neurons have
    # no such threshold.
    if case.get("neuron", "LIF") in SPIKING:
        return {"rel": 2.4e-3, "max": 0.02}
    return {"rel": 2e-6, "max": 1e-5}
