"""Launches that update neurons behind the product that forms their currents, a lane per neuron.

The encoders of a model are matrices that nothing writes.  `lay_out` gives a launch of
`hipra_gemv.fuse_lif` (and what `fuse_input_sums`, `fuse_learning` made of it) copies of its matrices in
the order in which a wave of csrc/gemv_lanes.hip reads them, and has it run that kernel instead.  Same sums in
the same order (the reference: clra_gemv.py:1043-1058, :1148-1153), same results.
"""

import numpy as np

from .hipra_gemv import N_DIES, _span, formed_sums, lay_out_matrices, spread_over_dies
from .hipra_sequence import _conflict
from .hipraggedarray import empty_device, to_device

WAVE, WG = 64, 256
MAX_COLS = 128      # one tile of the reference's order
RAW_COLS = 4        # matrices of so many columns are read as they lie in the signal buffer
PARTS = 4           # of an input sum are read together
TASK_WORDS = 40
_LIF, _NEURON = 1, 3  # EPI_LIF, EPI_NEURON
PAST_CACHE = 16     # NHIP_LANES_PAST_CACHE
# Bytes that the launches of a step move through the memory-side cache (256 MB), from which on it keeps too little of
# the matrices until the next step: they are read with non-temporal loads then.  Both sides stand at the kernel; they
# cross between 317 MB (256 x 4096 x 64: 57.7 / 61.1 us a step) and 350 (1000 x 4096 x 16: 94.5 / 86.8; 288 x 4096 x
# 64: 71.8 / 67.8), with a decoder for each of four connections between 303 (192 ensembles: 55.8 / 59.5) and 401 (256:
# 80.9 / 75.0).  Launches that visit active columns only count a tenth (populations spike in 8 to 11 % of the steps),
# those of csrc/gemv_tile.hip, whose loads are non-temporal, only where they write matrices: every column of 256 x
# 4096 x 64 multiplied 92.1 / 96.6, 320 of them 124.2 / 118.2; rate neurons 272 x 4096 x 64 94.6 / 96.3, 330 of them 122.0 /
# 114.7; PES 300 of 2000 x 32 128.1 / 119.0
STEP_BYTES, ACTIVE_SHARE = 330e6, 0.1
_KERNELS = {"nhip_gemv_%s_%s" % k: _NEURON if k[1] == "neuron" else _LIF
            for k in [("tile", "lif"), ("tile", "lif_sums"), ("tile", "lif_deferred"), ("tile", "neuron"),
                      ("rows", "lif"), ("rows", "lif_sums"), ("rows", "neuron")]}


class _Launch:
    """The arguments of a launch of `hipra_gemv.fuse_lif` that both kernels have."""

    def __init__(self, plan):
        name, args = plan.kern.__name__, plan.args
        self.neurons = _KERNELS[name]
        self.large = "_tile_" in name
        # (vec, class, words | lpr, words, items, coefs, dots, tasks, n, A, X, Yin, Y, pops, dt, upsample, V, W, S, ...)
        k = 8 if self.large else 7
        self.A, self.X = args[k:k + 2]
        self.dt, self.upsample = args[k + 5:k + 7]
        rest = args[k + 10:]  # (N | TAU, REF, AMP), then parts (large), or ranges and parts (small)
        n_states = 4 if self.neurons == _NEURON else 3
        self.buffers = list(args[k:k + 4]) + list(args[k + 7:k + 7 + n_states])
        if self.neurons == _NEURON:
            self.params, rest = (None, None, None), rest[1:]
        else:
            self.params, rest = rest[:3], rest[3:]
        self.deferred = getattr(plan, "host_deferred", None)
        if name.endswith("deferred"):
            self.buffers.append(rest[-1])
        self.parts = getattr(plan, "host_parts", None)
        self.ranges = getattr(plan, "host_ranges", None)
        has_parts = bool(rest) and rest[0 if self.large else -1] is not None
        self.known = ((self.parts is not None) == has_parts and (self.large or (self.ranges is not None) == has_parts)
                      and (self.deferred is not None) == name.endswith("deferred"))


def _matrices(plan):
    """{(start, row stride, rows, columns): index} of the matrices of a launch that have to be laid out, or None where
    the kernel does not hold one."""
    prog = plan.prog
    out = {}
    # (small items with several dot products each, all of them narrow: 16 populations of 500 with 3, 7 and 13 of them 10.0
    # us a step as they lie / 10.3 in this kernel, 11.9 / 13.0, 18.8 / 20.1; large items 55.4 / 17.3)
    if plan.kernel_class[0] == 2 and 2 * sum(len(prog.geometry[b]["dots"]) > 1 for b in plan.members) > len(plan.members):
        return None
    for b in plan.members:
        g = prog.geometry[b]
        cols = [d["a_shape1"] for d in g["dots"]]
        if cols and not 1 <= min(cols) <= max(cols) <= MAX_COLS:
            return None
        if cols and max(cols) <= RAW_COLS:
            continue
        # (one dot product at a time: more than one is not what this kernel is for)
        if len(cols) > 1 and plan.kernel_class[0] == 2:
            return None
        for d in g["dots"]:
            out.setdefault((d["a_start"], d["a_stride0"], g["y_len"], d["a_shape1"]), d["a_j"])
    return out


def matrix_spans(plan):
    """Intervals of the signal buffer that hold the matrices `lay_out` would copy, or None where the launch does not
    qualify."""
    name = getattr(plan.kern, "__name__", "")
    if name not in _KERNELS or plan.laid_out is not None or plan.kernel_class[0] not in (2, 3) or not plan.members:
        return None
    if getattr(plan, "host_tasks", None) is None if plan.kernel_class[0] == 3 else (
            getattr(plan, "host_tables", None) is None):
        return None
    launch = _Launch(plan)
    if not launch.known or any(ptr is None or ptr.value != launch.X.value for ptr in launch.buffers):
        return None
    mats = _matrices(plan)
    if mats is None or not any(plan.prog.geometry[b]["dots"] for b in plan.members):
        return None
    return sorted({_span(plan.prog.A, a_j) for a_j in mats.values()} - {None})


def _item_records(plan, launch):
    """A task record per item (or sum) of the launch, its rows still to be divided."""
    records = []
    prog, pops = plan.prog, np.asarray(plan.host_pops)
    if launch.large:
        first_of = {}
        for i, row in enumerate(plan.host_tasks):
            first_of.setdefault((int(row[0]), int(row[4])), i)
        rows = [plan.host_tasks[i] for i in first_of.values()]
    else:
        items, coefs = plan.host_tables[:2]
        rows = []
        for b in list(plan.members) + list(getattr(plan, "spare_items", ())):
            row = np.zeros(24, dtype=np.int32)
            row[0], row[4:12], row[12:15] = b, items[b], coefs[b, :3].view(np.int32)
            row[11] = 0
            if launch.ranges is not None:
                row[3], row[11] = launch.ranges[b]
            rows.append(row)
    for row in rows:
        b = int(row[0])
        record = np.zeros(TASK_WORDS, dtype=np.int32)
        record[:24] = row
        if launch.parts is None:
            record[3] = record[11] = 0
        if b < len(pops):
            record[24:24 + pops.shape[1]] = pops[b]
        if launch.deferred is not None and b < len(launch.deferred):
            record[36:40] = launch.deferred[b]
        records.append(record)
    return records


def sums_in_front(sum_plan, plan):
    """The input sums that the launch `sum_plan` right before `plan` forms, if `lay_out` can have the launch form them
    itself (`hipra_gemv.formed_sums`), or None.  Launches that read matrices as they lie form sums of up to 64
    elements for large matrices, of up to four for small ones; this kernel does of as many as it has columns
    (whole steps: 4 x 545 x 7 10.9 -> 8.7 us, 48 x 214 x 86 14.3 -> 10.3, 40 triples of 1028 x 7 20.3 ->
    17.9, 21 x 2381 x 94 with a population without input 24.0 -> 14.7)."""
    if (getattr(sum_plan, "name", "") != "hipra_gemv.wave_ref" or not hasattr(sum_plan, "prog")
            or sum_plan.prelude is not None or sum_plan.divided is not None or sum_plan.laid_out is not None
            or getattr(plan, "host_parts", None) is not None):
        return None
    carried = getattr(plan, "carried", None)  # (what rides in the launch has followed the sums so far)
    if carried is not None and any(_conflict(p, sum_plan) for p in carried.members):
        return None
    return formed_sums(sum_plan, plan, MAX_COLS)


def lay_out(plan, formed=None):
    """Make `plan` (for which `matrix_spans` gave spans, of constants) run the kernel with a lane per neuron, which forms
    the input sums `formed` (of `sums_in_front`) too.  The plan gets `lay_out_again`, for when the host has
    changed a matrix."""
    queue, lib, prog = plan.queue, plan.queue.lib, plan.prog
    launch = _Launch(plan)

    # the matrices, laid out
    mats = _matrices(plan)
    rows, cursor, at = [], 0, {}
    for key in mats:
        start, stride, M, N_cols = key
        quads = -(-N_cols // 4)
        at[key] = (cursor, quads)
        rows.append((start, stride, M, N_cols, cursor, quads, 0, 0))
        cursor += -(-M // WAVE) * quads
    if cursor >= 2 ** 31 // 256:  # (one buffer: as many elements as the signal buffer may have)
        return False
    dev_mats = to_device(queue, np.array(rows or [(0,) * 8], dtype=np.int32))
    dev_at = empty_device(queue, max(256 * cursor, 4))
    max_blocks = max([-(-r[2] // WAVE) for r in rows] + [1])

    # the tasks: up to 64 rows of an item from a multiple of 64 rows on
    pops = np.asarray(plan.host_pops)
    dots = prog.host_dots.copy()
    for b in plan.members:
        g = prog.geometry[b]
        for k, d in enumerate(g["dots"]):
            row = dots[first_dot(plan, b) + k]
            raw = max(e["a_shape1"] for e in g["dots"]) <= RAW_COLS
            row[5] = -1 if raw else 0  # (p0)
            if not raw:
                row[0], row[1] = at[d["a_start"], d["a_stride0"], g["y_len"], d["a_shape1"]]
    tasks, records = [], _item_records(plan, launch)
    where = {}
    if formed is not None:
        sums, spare = formed
        launch.parts = []
        for start, (_, parts) in sums.items():
            where[start] = (len(launch.parts), len(parts))
            launch.parts.extend(parts)
        launch.parts = np.array(launch.parts, dtype=np.int32)
        for start in spare:  # of an item without dot products and without neurons: Y = the sum
            record = np.zeros(TASK_WORDS, dtype=np.int32)
            record[0], record[3] = len(pops), where[start][0]
            record[4:12] = (start, 1, start, 1, 0, 0, sums[start][0], where[start][1])
            record[12] = np.float32(1).view(np.int32)
            records.append(record)
    for record in records:
        if record[9] > 0:
            record[16:24] = dots[record[8]]
            if int(record[19]) in where:
                record[3], record[11] = where[int(record[19])]
        M = int(record[10])
        many = np.repeat(record[None], -(-M // WAVE), axis=0)
        many[:, 1] = np.arange(len(many)) * WAVE
        many[:, 2] = np.minimum(WAVE, M - many[:, 1])
        tasks.append(many)
    tasks = spread_over_dies(np.concatenate(tasks))
    dev_parts = None
    if launch.parts is not None:  # every range padded with its last part: the kernel reads PARTS at a time
        padded, where = [], {}
        for i in np.flatnonzero(tasks[:, 11] > 0):
            key = (int(tasks[i, 3]), int(tasks[i, 11]))
            if key not in where:
                mine = launch.parts[key[0]:sum(key)].tolist()
                where[key] = len(padded)
                padded.extend(mine + mine[-1:] * (-len(mine) % PARTS))
            tasks[i, 3] = where[key]
        dev_parts = to_device(queue, np.array(padded, dtype=np.int32))
    tasks = for_the_dies(tasks)
    dev_tasks, dev_dots = to_device(queue, tasks), to_device(queue, dots)

    def again():
        lay_out_matrices(lib.nhip_lay_out_lanes, queue, dev_mats, len(rows), max_blocks, launch.A, dev_at)

    again()
    plan.lay_out_again = again
    carried = getattr(plan, "carried", None)
    old_size = plan.gsize[0] - (carried.gsize[0] if carried is not None else 0)
    plan.laid_out = (lib.nhip_gemv_lanes, (
        launch.neurons, dev_tasks.ptr, len(tasks), dev_dots.ptr, dev_at.ptr, launch.X, launch.dt, launch.upsample)
        + tuple(launch.params) + (dev_parts.ptr if dev_parts is not None else None, None))
    plan.full_args = tuple(plan.full_args) + (dev_mats, dev_at, dev_tasks, dev_dots, dev_parts)
    plan.gsize = (plan.gsize[0] - old_size + WG * (len(tasks) // (WG // WAVE)),)
    plan.host_tasks, plan.n_tasks = tasks[tasks[:, 2] > 0], len(tasks)
    plan.tag = "%s, laid out" % plan.tag

    def upload_pops():
        mine = (tasks[:, 2] > 0) & (tasks[:, 0] < len(pops))
        tasks[mine, 24:24 + pops.shape[1]] = np.asarray(plan.host_pops)[tasks[mine, 0]]
        dev_tasks.set(tasks.ravel())

    def leave_bits(mask):
        entry, args = plan.laid_out
        plan.laid_out = (entry, args[:-1] + (mask,))

    plan.upload_pops, plan.leave_bits = upload_pops, leave_bits
    return True


def read_past_the_cache(plans):
    """Launches of `lay_out` among the `plans` of a step that moves more than the memory-side cache keeps read their
    matrices past it."""
    share = lambda p: (ACTIVE_SHARE if getattr(p, "event_driven", False) else
                       0.0 if getattr(getattr(p, "kern", None), "__name__", "").startswith("nhip_gemv_tile")
                       and getattr(p, "laid_out", None) is None and not getattr(p, "learned_matrices", 0) else 1.0)
    moved = sum((getattr(p, "bw_per_call", None) or 0) * share(p) for p in plans)
    for plan in plans if moved > STEP_BYTES else ():
        if getattr(plan, "laid_out", None) is not None and plan.laid_out[0].__name__ == "nhip_gemv_lanes":
            entry, args = plan.laid_out
            plan.laid_out = (entry, (args[0] | PAST_CACHE,) + args[1:])


def for_the_dies(tasks):
    """The list of tasks with group g's four at 4 g, such that every die works through a contiguous range of the list
    given (the map of `nhip_xcd_remap`, made here once), filled up with tasks of no rows."""
    per_group = WG // WAVE
    groups = -(-len(tasks) // per_group)
    out = np.zeros((groups * per_group, tasks.shape[1]), dtype=np.int32)
    out[:len(tasks)] = tasks
    per, rem = divmod(groups, N_DIES)
    die, place = np.arange(groups) % N_DIES, np.arange(groups) // N_DIES
    at = np.where(die < rem, die * (per + 1), rem * (per + 1) + (die - rem) * per) + place
    return np.ascontiguousarray(out.reshape(groups, per_group, -1)[at].reshape(groups * per_group, -1))


def first_dot(plan, b):
    """Row of the table of dot products at which those of item `b` start."""
    starts = getattr(plan, "_first_dots", None)
    if starts is None:
        starts = np.concatenate([[0], np.cumsum([len(g["dots"]) for g in plan.prog.geometry])])
        plan._first_dots = starts
    return int(starts[b])
