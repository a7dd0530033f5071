"""The launch that decodes with matrices which an outer-product rule changes, in the form of csrc/gemv_learn.hip.

`lay_out` has a launch of `hipra_gemv.fuse_learning` (or of `fuse_hebbian`, which has that form already) read and
change its learned matrices a wave per row; what else it decodes, with matrices that nothing writes, visits the columns of the neurons that spiked only.  Same sums in the
same order (the reference: clra_gemv.py:1043-1058, :1148-1153; simulator.py:1334-1345), same results.
"""

import numpy as np

from .hipra_gemv import N_DIES, RULE_OUTER, _span, _spikes_item
from .hipraggedarray import empty_device, to_device

WG, ROWS, WAVE = 256, 4, 64


def _divided(plan):
    """(items with learned matrices, items that visit active columns, items whose rows are read whole) of a launch, or
    None where the kernel does not hold one."""
    learned, events, rows = [], [], []
    learns = set(plan.learn_of_item) if _from_tiles(plan) else set(
        plan.host_learn[1][plan.host_learn[0][:, 13] != 0].tolist())
    for b in plan.members:
        g = plan.prog.geometry[b]
        if len(g["dots"]) != 1 or g["y_len"] < 1:
            return None
        d = g["dots"][0]
        if d["a_shape1"] < 1 or (d["x_stride0"] != 1 and d["a_shape1"] > 1):
            return None
        (learned if b in learns else events if _spikes_item(plan.prog, b) else rows).append(b)
    groups = lambda items: sum(-(-plan.prog.geometry[b]["y_len"] // ROWS) for b in items)
    # (rows that are only read are what the kernel is not made for: as many as learned ones at most)
    if not learned or _from_tiles(plan) and groups(rows) > groups(learned):
        return None
    return learned, events, rows


def _from_tiles(plan):
    return getattr(plan.kern, "__name__", "") == "nhip_gemv_tile_filter_learn"


def matrix_spans(plan):
    """Intervals of the signal buffer that hold the matrices `lay_out` would copy, or None where the launch does not
    qualify."""
    if plan.laid_out is not None:
        return None
    if _from_tiles(plan):
        if getattr(plan, "filter_tables", None) is None or getattr(plan, "learn_of_item", None) is None:
            return None
        A, X, Yin, Y, F = plan.args[8:12] + (plan.filter_tables[2].ptr,)
    elif getattr(plan.kern, "__name__", "") == "nhip_gemv_learn" and getattr(plan, "host_learn", None) is not None:
        A, X, Yin, Y, _, F = plan.args[2:8]
    else:
        return None
    if any(ptr is None or ptr.value != X.value for ptr in (A, Yin, Y, F)):
        return None
    divided = _divided(plan)
    if divided is None or not (divided[1] or _from_tiles(plan)):
        return None
    return sorted({_span(plan.prog.A, plan.prog.geometry[b]["dots"][0]["a_j"]) for b in divided[1]} - {None})


def lay_out(plan):
    """Make `plan` (for which `matrix_spans` gave spans, of constants) run the kernel with a wave per learned row.  The
    plan gets `lay_out_again`, for when the host has changed a matrix."""
    from . import _lib

    queue, lib, prog = plan.queue, plan.queue.lib, plan.prog
    learned, events, rows = _divided(plan)
    bits = lambda v: int(np.float32(v).view(np.int32))
    coefs = lambda b: [bits(v) for v in (prog.alpha[b], prog.beta[b], prog.gamma[b])]
    if _from_tiles(plan):
        item_targets, dev_targets, F, host_targets = plan.filter_tables
        A, X, Yin, Y = plan.args[8:12]
        buffers, filters = (A, X, Yin, Y, dev_targets.ptr, F.ptr), (None, 0, None)
        tasks = []
        for b in learned + rows:
            g = prog.geometry[b]
            d = g["dots"][0]
            first, n = (int(v) for v in item_targets[b])
            target = [int(v) for v in host_targets[first][:4]] if n else [0] * 4
            rule = [0] * 8
            if b in plan.learn_of_item:
                e_start, f_start, alpha, _ = plan.learn_of_item[b]
                rule = [RULE_OUTER, f_start, e_start, 1, 0, 0, alpha, 0]
            for r in range(0, g["y_len"], ROWS):
                tasks.append([d["a_start"], d["a_stride0"], d["a_shape1"], d["x_start"], g["y_start"], g["y_stride0"],
                              g["y_in_start"], g["y_in_stride0"]] + coefs(b)
                             + [r, min(ROWS, g["y_len"] - r), int(b in plan.learn_of_item), first, n] + rule + target
                             + [0] * 4)
        tasks = np.array(tasks, dtype=np.int32)
    else:
        tasks, item_of, item_targets, host_targets = plan.host_learn
        tasks = tasks[~np.isin(item_of, events)]
        A = plan.args[2]
        buffers, filters = tuple(plan.args[2:8]), tuple(plan.args[8:11])
        if item_targets is None:
            item_targets = np.zeros((len(prog.geometry), 2), dtype=np.int32)
    # the groups of an item share its vectors: on one die (group g runs on die g % 8)
    per, rem = divmod(len(tasks), N_DIES)
    die, place = np.arange(len(tasks)) % N_DIES, np.arange(len(tasks)) // N_DIES
    tasks = np.ascontiguousarray(tasks[
        np.where(die < rem, die * (per + 1), rem * (per + 1) + (die - rem) * per) + place])

    by_matrix = {}
    for b in events:
        d = prog.geometry[b]["dots"][0]
        by_matrix.setdefault((d["a_start"], d["a_stride0"], prog.geometry[b]["y_len"], d["a_shape1"]), []).append(b)
    mats, records, cursor = [], [], 0
    for (start, stride, M, N), items in by_matrix.items():
        mp = -(-M // 16) * 16
        first_record = len(records)
        for b in items:
            g = prog.geometry[b]
            first, n = (int(v) for v in item_targets[b])
            target = [int(v) for v in host_targets[first][:4]] if n else [0] * 4
            for row0 in range(0, M, WAVE):  # a group per 64 rows
                records.append([cursor, mp, min(WAVE, M - row0), N, g["dots"][0]["x_start"], g["y_start"],
                                g["y_stride0"], g["y_in_start"], g["y_in_stride0"]] + coefs(b)
                               + [first, n, row0, 0] + target + [0] * 12)
        mats.append([start, stride, M, N, cursor, mp, first_record, len(records) - first_record])
        cursor += N * mp
    # (offsets inside a copy are 32-bit, in bytes)
    if cursor >= 2 ** 31 or len(mats) > 65535 or any(m[3] * m[5] >= 2 ** 30 for m in mats):
        return False
    records = np.array(records or [[0] * 32], dtype=np.int32)
    n_records = len(records) if events else 0
    plan.host_learned = (tasks, records[:n_records])
    dev_tasks, dev_records = to_device(queue, tasks), to_device(queue, records)
    dev_mats = to_device(queue, np.array(mats or [[0] * 8], dtype=np.int32))
    dev_at = empty_device(queue, max(cursor, 4))
    max_cols = max([m[3] for m in mats] + [1])

    def again():
        dev_records.set(records.ravel())
        _lib.check(lib.nhip_lay_out_columns(queue.handle, dev_mats.ptr, len(mats), max_cols, A, dev_at.ptr,
                                            dev_records.ptr), "laying out matrices")

    again()
    plan.lay_out_again = again
    carried = getattr(plan, "carried", None)
    plan.laid_out = (lib.nhip_gemv_learn_events, (
        dev_tasks.ptr, len(tasks)) + buffers + filters + (dev_records.ptr, n_records, dev_at.ptr))
    plan.full_args = tuple(plan.full_args) + (dev_tasks, dev_records, dev_mats, dev_at)
    plan.gsize = (WG * (len(tasks) + n_records) + (carried.gsize[0] if carried is not None else 0),)
    plan.lsize = (WG,)
    plan.tag = "%s, laid out" % plan.tag
    # (where populations spike densely, listing columns costs more than reading rows: their products are planned
    # again without, `Simulator._calibrate_event_launches`)
    plan.event_driven = n_records > 0
    return True
