"""Small networks: the whole plan list of a timestep as one resident launch.

The reference launches every plan of every step (plan.py:137-149); the executor here replays them as a
graph, in which a step of a small network still costs what its launches cost (4-5 us each).  For a network
whose signals and work lists fit the LDS of a compute unit, `resident_program` translates the plan
list into operations on an LDS image (csrc/resident.hip): one work-group runs all steps of a call
there, with the block functions of the ordinary launches, and the same results.
"""

import numpy as np

from . import hipra_sequence as seq
from .hipraggedarray import to_device
from .plan import Plan

WAVE, WAVES = 64, 8
LDS_WORDS = 39 * 1024  # RES_LDS_WORDS
ROWS4, ROWS1, LONG = 16, 32, 48  # kinds of csrc/resident.hip, + epilogue
LIF, DECODE, FILTER = 64, 65, 66
EPI_NONE, EPI_LIF, EPI_NEURON, EPI_FILTER = 0, 1, 3, 4
MAX_STEPS = 4096  # steps of one launch
# us of a step that one short launch of a replayed graph takes (two launches: 8.4-8.9 us for two populations,
# 10.6-11.5 for networks of a few thousand neurons)
GRAPH_LAUNCH = 4.2

OP_DTYPE = np.dtype([("kind", "<i4"), ("n_tasks", "<i4"), ("first", "<i4"), ("last", "<i4"),
                     ("n_rows", "<i4"), ("lanes", "<i4"), ("i0", "<i4"), ("upsample", "<i4"),
                     ("stride", "<i4"), ("pad", "<i4"), ("p", "<i4", (8,)), ("d0", "<f8"),
                     ("global", "<u8"), ("q", "<i4", (4,)), ("pad2", "<i4", (2,))])
SPAN_DTYPE = np.dtype([("ptr", "<u8"), ("words", "<i4"), ("lds", "<i4"), ("write_back", "<i4"), ("pad", "<i4")])
assert OP_DTYPE.itemsize == 112 and SPAN_DTYPE.itemsize == 24


class _Unfit(Exception):
    """The network has a part that the resident launch does not hold."""


class _Image:
    """Device arrays mirrored in LDS, and where."""

    def __init__(self, queue):
        self.queue, self.spans, self.words, self.keep = queue, {}, 0, []

    def add(self, ptr, words, write_back=False):
        address = ptr if isinstance(ptr, int) else int(ptr.value)
        if address % 16:
            raise _Unfit("an array that does not start on 16 bytes")
        end = address + 4 * words
        for start, (n, lds, _) in self.spans.items():
            if start <= address and end <= start + 4 * n and address < start + 4 * n:
                self.spans[start][2] |= write_back
                return lds + (address - start) // 4
            if address < start + 4 * n and start < end:  # (two copies, one of which would go stale)
                raise _Unfit("overlapping arrays")
        lds = self.words
        self.spans[address] = [int(words), lds, bool(write_back)]
        self.words += -(-int(words) // 4) * 4
        if self.words > LDS_WORDS:
            raise _Unfit("more than the LDS holds")
        return lds

    def table(self, array):
        """Upload a host table and mirror it."""
        array = np.ascontiguousarray(array, dtype=np.int32)
        if array.size == 0:
            array = np.zeros(4, dtype=np.int32)
        dev = to_device(self.queue, array.ravel())
        self.keep.append(dev)
        return self.add(dev.ptr, array.size)

    def lookup(self, address):
        """Word offset of an address inside a mirrored array."""
        for start, (n, lds, _) in self.spans.items():
            if start <= address < start + 4 * n:
                return lds + (address - start) // 4
        raise _Unfit("a pointer outside the mirrored arrays")


def _rows_ops(image, plan, sig_ptr, sig_lds):
    """Operations of one GEMV launch (small-item kernel, any epilogue)."""
    prog = plan.prog
    if plan.kernel_class[0] != 2 or getattr(plan, "host_tables", None) is None or any(
            ra.ptr.value != sig_ptr for ra in (prog.A, prog.X, prog.Y, prog.Y_in)):
        raise _Unfit("a product of another kind: %s" % plan.name)
    items, coefs = plan.host_tables[:2]
    kern = getattr(plan.kern, "__name__", "")
    ids = list(plan.members) + list(getattr(plan, "spare_items", ()))
    epi, q, i0, d0, upsample = EPI_NONE, [0, 0, 0, 0], 0, 0.0, 1
    pops = targets = None
    if kern in ("nhip_gemv_rows_lif", "nhip_gemv_rows_lif_sums", "nhip_gemv_rows_neuron"):
        epi = EPI_NEURON if kern.endswith("neuron") else EPI_LIF
        pops = np.asarray(plan.host_pops)
        if epi == EPI_LIF and np.any(pops[ids, 7] & 7):
            raise _Unfit("a neuron parameter per neuron")
        d0, upsample = float(plan.args[12]), int(plan.args[13])
        states = [a.value for a in plan.args[14:17 if epi == EPI_LIF else 18] if a is not None]
        if any(a != sig_ptr for a in states):
            raise _Unfit("neuron states in another array")
        ranges = getattr(plan, "host_ranges", None)
        if (ranges is None) != (kern == "nhip_gemv_rows_lif" or plan.args[-1] is None):
            raise _Unfit("input sums without their ranges")
        q[0] = image.table(pops)  # (small: words of an item that no task needs cost nothing)
        if ranges is not None:
            i0, q[1], q[2] = 1, image.table(plan.host_parts), image.table(ranges)
    elif kern == "nhip_gemv_rows_filter":
        epi = EPI_FILTER
        item_targets, dev_targets, F, targets = plan.filter_tables
        if F.ptr.value != sig_ptr:
            raise _Unfit("filter outputs in another array")
        q[0], q[2] = image.table(targets), image.table(item_targets)
    elif kern != "nhip_gemv":
        raise _Unfit("a launch of another kind: %s" % kern)
    dots, shared = prog.host_dots, []
    wave_tasks, long_tasks, row_tasks, lif_tasks, decode_rows = [], [], [], [], []
    floats = lambda *v: tuple(int(x) for x in np.array(v, dtype=np.float32).view(np.int32))
    dt_inv = np.float32(1.0 / d0) if d0 else np.float32(0)
    for b in ids:
        rows, n_dots = int(items[b, 6]), int(items[b, 5])
        mine = dots[items[b, 4]:items[b, 4] + n_dots]
        y_start, y_stride, yin, yin_stride = (int(v) for v in items[b, :4])
        if epi == EPI_LIF and int(pops[b, 7]) & 256 and y_stride == 1 and rows >= 8 and (
                n_dots == 0 or n_dots == 1 and int(mine[0, 2]) <= 4) and not (
                    n_dots == 0 and ranges is not None and int(ranges[b, 1]) > 0):
            a, a_stride, n_cols, x, x_stride = (int(v) for v in mine[0, :5]) if n_dots else (0, 0, 0, 0, 0)
            first, n_parts = (int(v) for v in ranges[b]) if n_dots and ranges is not None else (0, 0)
            amp = pops[b, 6:7].view(np.float32)[0]
            for r in range(0, rows, WAVE):
                lif_tasks.append((min(WAVE, rows - r), n_cols, yin + r * yin_stride, yin_stride, a + r * a_stride,
                                  a_stride, x, x_stride) + floats(*coefs[b, :3]) + (int(pops[b, 4]), int(pops[b, 5]))
                                 + floats(amp * dt_inv)
                                 + (-1 if int(pops[b, 7]) & 1024 else y_start + r, int(pops[b, 0]) + r,
                                    int(pops[b, 1]) + r, int(pops[b, 2]) + r, first, n_parts, int(r == 0), 0, 0, 0))
            continue
        # (rows of a launch with neurons that drive none, and are no sums of parts, are plain rows)
        plain = epi in (EPI_NONE, EPI_FILTER) or (
            not int(pops[b, 7 if epi == EPI_LIF else 10]) & 256 and (ranges is None or int(ranges[b, 1]) == 0))
        if plain and n_dots == 1 and int(mine[0, 2]) >= 1 and (
                int(mine[0, 4]) == 1 or int(mine[0, 2]) == 1) and (
                    rows < 8 or int(mine[0, 2]) > 4) and (int(mine[0, 2]) < 256 or epi not in (EPI_NONE, EPI_FILTER)):
            first, n_targets = (int(v) for v in item_targets[b]) if targets is not None else (0, 0)
            a, a_stride, n_cols, x, _ = (int(v) for v in mine[0, :5])
            for r in range(rows):
                decode_rows.append((a + r * a_stride, x, n_cols, y_start + r * y_stride, yin + r * yin_stride,
                                    first, n_targets, r) + floats(*coefs[b, :3]) + (0,))
            continue
        record = np.zeros(16, dtype=np.int32)
        record[0], record[4:12], record[12:15] = b, items[b], coefs[b, :3].view(np.int32)
        if pops is not None:
            record[3], record[11], record[15] = (pops[b, 0], pops[b, 1], pops[b, 7]) if epi == EPI_LIF else (0, 0, 0)
        if targets is not None:
            record[3], record[11] = item_targets[b]
        if rows >= 8 and (n_dots == 0 or int(mine[:, 2].max()) <= 4):
            for r in range(0, rows, WAVE):
                record[1], record[2] = r, min(WAVE, rows - r)
                wave_tasks.append(record.copy())
        elif (epi in (EPI_NONE, EPI_FILTER) and n_dots and int(mine[:, 2].min()) >= 128
              and np.all(mine[:, 4] == 1)):
            for r in range(rows):
                record[1], record[2] = r, 1
                long_tasks.append(record.copy())
        else:
            row_tasks += [(b, r, 1, 0) for r in range(rows)]
    out = []

    def op(kind, tasks, n_tasks):
        row = np.zeros((), dtype=OP_DTYPE)
        own = kind in (LIF, DECODE)  # (work lists that need no table of the launch)
        row["kind"], row["n_tasks"], row["n_rows"], row["i0"] = kind if own else kind + epi, n_tasks, len(tasks), i0
        row["upsample"], row["d0"], row["q"] = upsample, d0, q
        table = image.table(np.array(tasks, dtype=np.int32))
        if own:
            row["p"][0], row["p"][4] = table, sig_lds
        else:
            if not shared:
                shared.extend([image.table(items), image.table(coefs.view(np.int32)), image.table(dots)])
            row["p"][:5] = tuple(shared) + (table, sig_lds)
        # (time of a task alone on its SIMD, us)
        if kind == DECODE:
            cost = 0.5 + 0.006 * max(t[2] for t in tasks)
        elif kind == LIF:
            # (alone 0.75, without sums; where every wave has some the two of a SIMD slow each other)
            n_parts = max(t[19] for t in tasks)
            cost = 1.35 + 0.03 * n_parts if n_parts else 0.93
        else:
            cost = (2.8 if epi == EPI_NEURON else 1.5) if kind == ROWS1 else 1.25
        out.append((row, cost))

    if lif_tasks:
        op(LIF, lif_tasks, len(lif_tasks))
    if decode_rows:
        op(DECODE, decode_rows, -(-len(decode_rows) // (WAVE // 4)))
    if wave_tasks:
        op(ROWS1, wave_tasks, len(wave_tasks))
    if long_tasks:
        op(LONG, long_tasks, len(long_tasks))
    if row_tasks:
        op(ROWS4, row_tasks, -(-len(row_tasks) // (WAVE // 4)))
    return out


# per kind of sequence operation: which pointers are work lists or data in LDS (the others stay where they are)
_GLOBAL_POINTER = {seq.SEQ_PRESENTINPUT: 3, seq.SEQ_PROBES: 5}


def _simple_filters(image, plan, sig_ptr, sig_lds):
    """First-order filters of vectors, an element per lane, or None where the launch holds others."""
    spec = getattr(plan, "lf_spec", None)
    if spec is None or getattr(plan, "higher_order", True):
        return None
    X, Y, A, B = (spec[k] for k in ("X", "Y", "A", "B"))
    if X.ptr.value != sig_ptr or Y.ptr.value != sig_ptr or int(X.sizes.sum()) > 512 or (
            np.any(X.shape1s != 1) or np.any(Y.shape1s != 1)):
        return None
    a_host, b_host = A.to_host(), B.to_host()
    rows = []
    for k in range(len(X)):
        a = np.float32(a_host[k][0, 0]) if int(A.shape0s[k]) else np.float32(np.nan)
        if int(A.shape0s[k]) and np.isnan(a):
            return None
        bits = tuple(int(v) for v in np.array([a, b_host[k][0, 0]], dtype=np.float32).view(np.int32))
        for i in range(int(X.shape0s[k])):
            rows.append((int(X.starts[k]) + i * int(X.stride0s[k]), int(Y.starts[k]) + i * int(Y.stride0s[k])) + bits)
    row = np.zeros((), dtype=OP_DTYPE)
    row["kind"], row["n_rows"], row["n_tasks"] = FILTER, len(rows), -(-len(rows) // WAVE)
    row["p"][0], row["p"][4] = image.table(np.array(rows, dtype=np.int32)), sig_lds
    return [(row, 0.25)]


def _sequence_op(image, plan, sizes):
    found = seq.sequence_op(plan)
    if found is None:
        raise _Unfit("a launch of another kind: %s" % plan.name)
    kind, n, lanes, i0, d0, pointers = found
    row = np.zeros((), dtype=OP_DTYPE)
    lanes = min(int(lanes), WAVE)
    row["kind"], row["n_rows"], row["lanes"], row["i0"], row["d0"] = kind, n, lanes, i0, d0
    row["n_tasks"] = -(-n // (WAVE // lanes))
    for k, ptr in enumerate(pointers):
        address = seq._addr(ptr)
        if k == _GLOBAL_POINTER.get(kind):
            row["global"] = address
        elif address:
            if address in sizes:
                # (what an operation may write: everything but work lists and coefficients)
                written = (kind, k) in ((seq.SEQ_LINEARFILTER, 1), (seq.SEQ_LINEARFILTER, 6),
                                        (seq.SEQ_LINEARFILTER, 7), (seq.SEQ_PROBES, 1), (seq.SEQ_PROBES, 2))
                row["p"][k] = image.add(address, sizes[address], write_back=written)
            else:
                row["p"][k] = image.lookup(address)
    return [(row, 0.4 + 0.1 * getattr(plan, "row_iterations", 1))]


def _arrays_of(plan):
    """{address: words} of the device arrays a plan keeps."""
    out = {}
    for a in plan.full_args:
        if hasattr(a, "ptr") and hasattr(a, "size") and a.ptr.value:
            out[int(a.ptr.value)] = int(a.size)
    return out


def _schedule(ops, memory):
    """Programs of the waves for the operations of every plan (``ops[i]``: list of (record, cost of a task))
    and what each plan reads and writes.

    A plan goes into the phase behind the last of the earlier plans it conflicts with; one that is a
    single task may follow a plan it conflicts with in the same phase, on the same wave, if that is the
    only wave of the phase it has to wait for.  In a phase the operations go to the waves with the least to do, an
    operation of many tasks to many.  Returns (a list of records per wave, estimated time of a step in us)."""
    if any(r is None or w is None for r, w in memory):
        raise _Unfit("a plan that does not say what it touches")
    single = [len(o) == 1 and int(o[0][0]["n_tasks"]) == 1 for o in ops]
    phase, strand = [], []  # of every plan: its phase, the single task at the head of its strand (or None)
    for i, (r, w) in enumerate(memory):
        wait = [j for j, (rj, wj) in enumerate(memory[:i]) if (wj & r) or (wj & w) or (rj & w)]
        last = max([phase[j] for j in wait] + [-1])
        heads = {strand[j] for j in wait if phase[j] == last}
        if last >= 0 and single[i] and len(heads) == 1 and None not in heads:
            phase.append(last)
            strand.append(heads.pop())
        else:
            phase.append(last + 1)
            strand.append(i if single[i] else None)
    programs, total = [[] for _ in range(WAVES)], 0.0
    for ph in range(max(phase) + 1):
        load = np.zeros(WAVES)
        here = [i for i in range(len(ops)) if phase[i] == ph]
        for head in sorted({strand[i] for i in here if strand[i] is not None}):
            wave = int(np.argmin(load))
            for i in here:
                if strand[i] == head:
                    (op, cost), = ops[i]
                    op["first"], op["stride"] = 0, 1
                    programs[wave].append(op.copy())
                    load[wave] += 0.2 + cost
        for i in here:
            if strand[i] is not None:
                continue
            for op, cost in ops[i]:
                n = int(op["n_tasks"])
                order = np.argsort(load, kind="stable")
                # as many waves as are no busier than the operation leaves the others
                best, k = None, 1
                for waves in range(1, min(n, WAVES) + 1):
                    trial = load.copy()
                    for q in range(waves):
                        trial[order[q]] += 0.2 + cost * -(-(n - q) // waves)
                    if best is None or trial.max() < best - 1e-9:
                        best, k = trial.max(), waves
                for q in range(k):
                    op["first"], op["stride"] = q, k
                    programs[order[q]].append(op.copy())
                    load[order[q]] += 0.2 + cost * -(-(n - q) // k)
        total += load.max() + 0.2
        for program in programs:
            if not program or int(program[-1]["last"]):  # nothing to do in this phase
                program.append(np.zeros((), dtype=OP_DTYPE))
            program[-1]["last"] = 1
    return programs, total


class Resident:
    """The launch of `n` steps (`__call__`)."""

    def __init__(self, queue, image, programs):
        spans = np.zeros(len(image.spans), dtype=SPAN_DTYPE)
        for row, (address, (words, lds, back)) in zip(spans, image.spans.items()):
            row["ptr"], row["words"], row["lds"], row["write_back"] = address, words, lds, back
        self.ops = np.array([op for program in programs for op in program], dtype=OP_DTYPE)
        self.first_op = np.concatenate([[0], np.cumsum([len(p) for p in programs])]).astype(np.int32)
        dev_spans, dev_ops = (to_device(queue, a.view(np.int32)) for a in (spans, self.ops))
        self.queue, self.n_words = queue, image.words
        self.args = (dev_spans.ptr, len(spans), dev_ops.ptr, self.first_op.ctypes.data, WAVES)
        self.keep = (dev_spans, dev_ops) + tuple(image.keep)

    def __call__(self, n):
        from . import _lib

        while n > 0:
            steps = min(n, MAX_STEPS)
            _lib.check(self.queue.lib.nhip_resident(self.queue.handle, *self.args, steps), "resident steps")
            n -= steps


def resident_program(queue, plans, all_data, n_launches):
    """`Resident` for the plan list of a step -- (plan, memory it reads, memory it writes) before short plans
    are merged and carried --, or None where it holds a plan of a kind the resident launch does not hold,
    does not fit the LDS, or would not be shorter than `n_launches` launches of a graph: by the costs
    of the operations in their wave, measured (csrc/resident.hip; the estimates of 28 networks between
    2.6 and 12.3 us lie at most 22 % above and 10 % below what they take).  Near the limit, with the launches of
    a graph beside it: two populations of 1,408 neurons 8.3 us a step (8.5), of 1,500 9.2 (8.8), four of 300 x 2
    with second-order synapses 8.5 (9.3), of 400 x 2 9.9 (9.7).  What copying the image in and out adds to a
    call needs no term: a call of one step takes 31 us with 8 KB of it and 40 with 100, a graph's 46-53."""
    memory = [(r, w) for _, r, w in plans]
    plans = [p for p, _, _ in plans]
    if not plans or not all(isinstance(p, Plan) for p in plans):
        return None
    image = _Image(queue)
    try:
        sig = image.add(all_data.ptr, all_data.dev_buf.size, write_back=True)
        ops = []
        for p in plans:
            if hasattr(p, "prog"):
                found = _rows_ops(image, p, all_data.ptr.value, sig)
            else:
                found = _simple_filters(image, p, all_data.ptr.value, sig)
                if found is None:
                    found = _sequence_op(image, p, _arrays_of(p))
            ops.append(found)
        programs, estimate = _schedule(ops, memory)
    except _Unfit:
        return None
    program = Resident(queue, image, programs)
    program.estimate = estimate
    return program if estimate < GRAPH_LAUNCH * n_launches else None
