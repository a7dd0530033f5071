"""Products with constant matrices, each output row with the filters it feeds, from copies of the matrices in
the order in which csrc/gemv_dots.hip reads them: decoders, transforms.

`lay_out` has a launch of `hipra_gemv` (small items, long rows, large items, columns of the neurons that spiked; with
or without the filters of `fuse_linearfilter`) run that kernel instead.  Same sums in the same order (the reference:
clra_gemv.py:1043-1058, :1148-1153), same results.
"""

import numpy as np

from .hipra_gemv import GROUP_ROW_MIN_COLS, GROUP_ROWS_MAX, STREAM_FLAT, _span, lay_out_matrices
from .hipraggedarray import empty_device, to_device

WG, TILE = 256, 128
ROW_COLS = 256  # rows of up to so many columns have a record each, longer ones share one
# ... but few long rows take a group each elsewhere (`GROUP_ROWS_MAX` of hipra_gemv): 10 rows of 9,216 columns, whole
# steps 25.9 us; with a group per row and their vector through LDS 26.5
# Launches that visit active columns only, up to so many bytes of copies: beyond, the columns that count are fewer
# bytes than the matrices, which the L2 of the dies no longer hold.  Whole steps, active columns / all of them:
# 20 x 32 x 600 (1.9 MB) 9.5 / 7.9 us, 100 x 16 x 1000 (6.5) 7.6 / 7.6, 37 x 50 x 1501 (15) 10.6 / 10.1,
# 12 x 64 x 5000 (19; a group per item) 16.7 / 14.1, 60 x 30 x 3000 (30) 14.1 / 16.8
EVENT_MAX_BYTES = 20 << 20
# Other launches, up to so many: beyond, encoders and decoders of a step no longer stay in the memory-side cache (256 MB),
# and non-temporal rows in long runs come faster. Rate neurons, whole steps, this kernel / csrc/gemv_tile.hip:
# 84 MB of decoders (80 x 64 x 4096) 32.0 / 34.6 us, 134 MB 48.0 / 53.3, 168 MB 65.5 / 59.1, 268 MB 101 / 89
MAX_BYTES = 144 << 20
GROUPS_FOR_FEW_ROWS = 2048  # of groups that are mostly empty
# Rows of up to 256 columns are padded to 32, 64, 128 or 256 of them, as the launch's widest, and have records of 64
# bytes.  `_reads_little` says where that pays; what it says no to reads its matrices as they lie.  Whole steps, as
# they lie / laid out:
# - small items (four lanes or one per row), up to four columns: 90,000 x 2 11.9 / 11.9 us, 130,000 x 1 11.7 / 12.4,
#   200,000 x 2 12.6 / 17.2, 1,000,000 x 2 20.8 / 42.1; from five columns on 4,000 of 50 x 5 18.4 / 17.3, 8,000 of
#   50 x 32 38.7 / 28.2; rows widened by others of the launch: 100 of 50 x 2 beside 10 x 100 11.0 / 11.7, 1,000 of them
#   12.8 / 14.8 (beside 10 x 250 14.2 / 22.1; 100 of them 12.9 / 11.9)
# - large items: what is read fits the L2 of the dies (32 MB): 65,000 x 16 12.3 / 8.8, 130,000 x 32 15.9 / 12.7; beyond,
#   200,000 x 8 14.4 / 17.3, x 32 17.2 / 19.8, x 64 19.2 / 18.2, x 100 28.7 / 25.9, 400,000 x 40 26.9 / 28.3, 130,000 x
#   68 19.1 / 20.2, x 132 26.6 / 31.5; rows that are not on 16-byte boundaries 200,000 x 15 16.2 / 17.5, x 50 20.4 /
#   18.0, x 66 41.8 / 26.1
# - ... without filters, where rows as they lie are read faster: 40,000 x 128 20.1 / 16.6, 32 of 2000 x 128 22.1 / 24.4,
#   80 of 2000 x 51 23.4 / 25.4, 64,000 x 200 25.9 / 29.3, 8 of 8000 x 256 26.1 / 28.0; not on 16-byte boundaries 40 of
#   2000 x 66 28.0 / 25.6
# Longer rows of up to 144 MB (250 to 1,700 columns, padded to twice that at most) are faster laid out throughout
SMALL_ITEMS_BYTES, L2_BYTES = 20 << 20, 32 << 20


class _Launch:
    def __init__(self, plan):
        name, args = getattr(plan.kern, "__name__", ""), plan.args
        self.known = name in ("nhip_gemv", "nhip_gemv_rows_filter", "nhip_gemv_tile", "nhip_gemv_tile_filter",
                              "nhip_gemv_events") and hasattr(plan, "prog") and plan.laid_out is None
        if not self.known:
            return
        self.events = name == "nhip_gemv_events"
        self.order, self.item_targets, self.targets, F = 1, None, None, None
        if self.events:
            self.A, (self.X, Yin, Y) = plan.prog.A.ptr, args[3:6]
            filtered = args[6] is not None
        else:
            k = 7 if name == "nhip_gemv_rows_filter" else 8 if "_tile" in name else 9
            self.A, self.X, Yin, Y = args[k:k + 4]
            filtered = name.endswith("_filter")
            self.known = "_tile" in name or name != "nhip_gemv" or args[0] == 2
        if filtered:
            tables = getattr(plan, "filter_tables", None)
            if tables is None:
                self.known = False
                return
            self.item_targets, self.targets, F, self.host_targets = tables
            self.order = int(args[8] if self.events else args[-1])
        self.buffers = [self.A, Yin, Y] + ([F.ptr] if F is not None else [])


def _shape(plan):
    """(tiles, quads) of the kernel for a launch, or None where it holds none or has nothing to give."""
    g = [plan.prog.geometry[b] for b in plan.members]
    if not g or any(len(item["dots"]) != 1 or item["dots"][0]["a_shape1"] < 1 for item in g):
        return None
    dots = [item["dots"][0] for item in g]
    cols = max(d["a_shape1"] for d in dots)
    if cols <= ROW_COLS:
        if any(d["x_stride0"] != 1 and d["a_shape1"] > 1 for d in dots):
            return None
        quads = -(-cols // 16)
        return (2, 8) if cols > TILE else (1, 2 if quads <= 2 else 4 if quads <= 4 else 8)
    rows = sum(item["y_len"] for item in g)
    tiles = 4 if cols <= 4 * TILE else 8 if cols <= 8 * TILE else 16
    if cols >= GROUP_ROW_MIN_COLS and rows <= GROUP_ROWS_MAX:
        return None
    per_group = WG // (4 * tiles)
    groups = sum(-(-item["y_len"] // per_group) for item in g)
    if groups > GROUPS_FOR_FEW_ROWS and 4 * rows < groups * per_group:
        return None
    return tiles, 8


def _copy_units(plan, tiles, quads):
    """{matrix: 64-byte units of its copy}"""
    out = {}
    for b in plan.members:
        g = plan.prog.geometry[b]
        d = g["dots"][0]
        passes = -(-d["a_shape1"] // (tiles * TILE))
        out[d["a_start"], d["a_stride0"], g["y_len"], d["a_shape1"]] = (passes * quads * tiles, d["a_j"])
    return out


def _reads_little(plan, filtered, tiles, quads, mats):
    """Is what the kernel reads of its copies and records little enough, against the matrices as they lie?"""
    if tiles > 2:
        return True
    kind, cols = tuple(plan.kernel_class), max(key[3] for key in mats)
    read = sum(64 * key[2] * (units + 1) for key, (units, _) in mats.items())
    useful = sum(4 * key[2] * key[3] for key in mats)
    if kind[0] == 2:
        own = sum(64 * key[2] * ((2 if key[3] <= 32 else 4 if key[3] <= 64 else 8 if key[3] <= TILE else 16) + 1)
                  for key in mats)
        if read > 2 * own:
            return cols > TILE and read <= SMALL_ITEMS_BYTES
        return read <= max(10 * useful, SMALL_ITEMS_BYTES)
    if read <= L2_BYTES or kind == (3, 0, 1):
        return True
    if not filtered:
        return False
    if kind == (3, STREAM_FLAT, 4):
        return cols > 16
    return cols > 32 and (2 * read <= 3 * useful or (read - useful <= L2_BYTES and 2 * read <= 5 * useful))


def matrix_spans(plan):
    """Intervals of the signal buffer that hold the matrices `lay_out` would copy, or None where the launch does not
    qualify."""
    launch = _Launch(plan)
    if not launch.known or any(ptr is None or ptr.value != launch.X.value for ptr in launch.buffers):
        return None
    shape = _shape(plan)
    if shape is None:
        return None
    mats = _copy_units(plan, *shape)
    size = sum(64 * key[2] * units for key, (units, _) in mats.items())
    if size > (EVENT_MAX_BYTES if launch.events else MAX_BYTES) or not _reads_little(
            plan, launch.targets is not None, *shape, mats):
        return None
    return sorted({_span(plan.prog.A, a_j) for _, a_j in mats.values()} - {None})


def lay_out(plan):
    """Make `plan` (for which `matrix_spans` gave spans, of constants) run the kernel that reads copies of its
    matrices.  The plan gets `lay_out_again`, for when the host has changed a matrix."""
    queue, lib, prog = plan.queue, plan.queue.lib, plan.prog
    launch = _Launch(plan)
    tiles, quads = _shape(plan)
    mats, at, rows, cursor = _copy_units(plan, tiles, quads), {}, [], 0
    for key, (units, _) in mats.items():
        at[key] = (cursor, units)
        rows.append(key + (cursor, 4 * tiles, quads, units))
        cursor += key[2] * units
    dev_mats = to_device(queue, np.array(rows, dtype=np.int32))
    dev_at = empty_device(queue, 16 * cursor)
    max_rows = max(r[2] for r in rows)
    bits = lambda v: int(np.float32(v).view(np.int32))
    per_group = WG // (4 * tiles)
    records, item_of = [], []
    full, most = 32, 0
    for b in plan.members:
        g, d = prog.geometry[b], prog.geometry[b]["dots"][0]
        M, N = g["y_len"], d["a_shape1"]
        start, units = at[d["a_start"], d["a_stride0"], M, N]
        first, n_targets = (0, 0) if launch.item_targets is None else (int(v) for v in launch.item_targets[b])
        target = [int(v) for v in launch.host_targets[first][:4]] if n_targets else [0] * 4
        coefs = [bits(v) for v in (prog.alpha[b], prog.beta[b], prog.gamma[b])]
        if tiles <= 2:
            full = min([full] + [max(0, min(TILE, N - TILE * t) // 4) for t in range(tiles)])
            most = max(most, -(-min(N, TILE) // 4))
            r = np.arange(M)
            mine = np.empty((M, 16), dtype=np.int32)
            mine[:] = [start, d["x_start"], N, n_targets, g["y_start"], g["y_in_start"], first, 0] + coefs + [0] + target
            mine[:, [0, 4, 5, 7]] += np.stack([r * units, r * g["y_stride0"], r * g["y_in_stride0"], r], 1).astype(np.int32)
        else:
            r = np.arange(0, M, per_group)
            mine = np.empty((len(r), 32), dtype=np.int32)
            mine[:] = [start, units, N, d["x_start"], d["x_stride0"], 0, 0, n_targets, g["y_start"], g["y_stride0"],
                       g["y_in_start"], g["y_in_stride0"]] + coefs + [first] + target + [0] * 12
            mine[:, 5], mine[:, 6] = r, np.minimum(per_group, M - r)
        records.append(mine)
        item_of.append(np.full(len(mine), b))
    if tiles <= 2:  # whole groups: more of the last row, that store nothing
        pad = np.repeat(records[-1][-1:], -sum(map(len, records)) % per_group, axis=0)
        pad[:, 3] = -1
        records.append(pad)
    records, item_of = np.concatenate(records), np.concatenate(item_of)
    n_groups = len(records) // per_group if tiles <= 2 else len(records)
    dev_records = to_device(queue, records)

    def again():
        lay_out_matrices(lib.nhip_lay_out_dots, queue, dev_mats, len(rows), max_rows, launch.A, dev_at)

    again()
    plan.lay_out_again = again
    carried = getattr(plan, "carried", None)
    plan.laid_out = (lib.nhip_gemv_dots, (
        tiles, quads, launch.order, dev_records.ptr, n_groups, dev_at.ptr, launch.X,
        launch.targets.ptr if launch.targets is not None else dev_records.ptr, full if tiles <= 2 else 0, most))
    plan.full_args = tuple(plan.full_args) + (dev_mats, dev_at, dev_records)
    plan.gsize = (WG * n_groups + (carried.gsize[0] if carried is not None else 0),)
    plan.lsize = (WG,)
    plan.tag = "%s, laid out" % plan.tag
    plan.host_records = records

    def upload_x_bits():
        """The spikes of some items are bits now (`hipra_gemv.store_spikes_as_bits`)."""
        value = dict(zip(plan.event_record_item.tolist(), plan.event_table[:, 15].tolist()))
        records[:, 20] = [value[b] for b in item_of.tolist()]
        dev_records.set(records.ravel())

    plan.upload_x_bits = upload_x_bits
    return True
