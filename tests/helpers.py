"""Shared helpers for the parity tests."""

import numpy as np

from nengo_ocl_amd.raggedarray import RaggedArray


def RA(arrays, dtype=np.float32, **kw):
    return RaggedArray(arrays, dtype=dtype, **kw)


def clone(ra):
    """An independent host copy (same metadata, own buffer)."""
    return RaggedArray.from_buffer(
        np.array(ra.buf), ra.starts, ra.shape0s, ra.shape1s, ra.stride0s, ra.stride1s, names=ra.names
    )


def to_dev(queue, ra):
    from nengo_ocl_amd.hipraggedarray import HIPRaggedArray

    return HIPRaggedArray(queue, ra)


def host_queue(monkeypatch):
    """A queue whose arrays lie in host memory and whose launches do nothing: plans can be made and
    looked at without a device."""
    import contextlib
    import ctypes
    import types

    import torch
    from nengo_ocl_amd import _lib, hipraggedarray

    real = _lib.lib()
    host_functions = ("nhip_gemv_tile_rows", "nhip_gemv_rows_per_task", "nhip_conv2d_groups")

    class Lib:
        def __getattr__(self, name):
            if name in host_functions:
                return getattr(real, name)
            launch = lambda *args: 0
            launch.__name__ = getattr(real, name).__name__
            return launch

    monkeypatch.setattr(hipraggedarray, "_TORCH", torch)
    return types.SimpleNamespace(
        lib=Lib(), handle=ctypes.c_void_p(1), device=torch.device("cpu"), arch="gfx950", n_compute_units=256,
        global_mem_size=288 << 30, stream=types.SimpleNamespace(synchronize=lambda: None),
        finish=lambda: None, context=contextlib.nullcontext, read=lambda words: words.numpy().copy())


def host_simulators(monkeypatch):
    """Simulators on queues of that kind: their plan lists can be looked at, steps compute nothing."""
    import torch
    from nengo_ocl_amd import hipraggedarray

    monkeypatch.setattr(hipraggedarray, "Queue", lambda device=0: host_queue(monkeypatch))
    for name in ("empty", "zeros"):
        make = getattr(torch, name)
        monkeypatch.setattr(torch, name, lambda *a, pin_memory=False, _make=make, **k: _make(*a, **k))


def run_plans(plans):
    for p in plans:
        p()


PHILOX_KNOWN_ANSWERS = [
    # counter, key -> output: the generator's published test vectors (Random123 kat_vectors,
    # philox4x32 with 10 rounds)
    ([0, 0, 0, 0], [0, 0], [0x6627e8d5, 0xe169c58d, 0xbc57ac4c, 0x9b00dbd8]),
    ([0xffffffff] * 4, [0xffffffff] * 2, [0x408f276d, 0x41c83b0e, 0xa20bc7c6, 0x6d5451fd]),
    ([0x243f6a88, 0x85a308d3, 0x13198a2e, 0x03707344], [0xa4093822, 0x299f31d0],
     [0xd16cfe09, 0x94fdcceb, 0x5001e420, 0x24126ea1]),
]


def buffer_differences(sim_a, sim_b, limit=12):
    """Where the signal buffers of two simulators of one model differ: a list of
    ``(signal name, number of differing elements, largest difference, first index)``,
    empty when every float has the same value (NaNs in the same places count as equal)."""
    # (the buffer as the host is shown it: currents that are not stored brought up to date,
    # signals that device memory holds a step ahead taken from their copy)
    a, b = sim_a.signal_buffer(), sim_b.signal_buffer()
    if a.shape != b.shape:
        return [("buffer sizes", a.size, b.size, -1)]
    bad = ~((a == b) | (np.isnan(a) & np.isnan(b)))
    if not bad.any():
        return []
    ra = sim_b.all_data
    out = []
    for i, base in enumerate(sim_b.all_bases):
        start = int(ra.starts[i])
        n = int(ra.shape0s[i]) * int(ra.shape1s[i])
        where = np.flatnonzero(bad[start:start + n])
        if len(where):
            diff = np.abs(a[start:start + n][where].astype(np.float64) - b[start:start + n][where])
            out.append((str(getattr(base, "name", i)), len(where), float(np.nanmax(diff)),
                        int(where[0])))
            if len(out) >= limit:
                break
    return out or [("outside every base", int(bad.sum()), 0.0, int(np.flatnonzero(bad)[0]))]


def assert_same_signals(sim_a, sim_b):
    """Every signal of the two simulators holds the same values; a failure names the
    signals that differ instead of printing two buffers."""
    diffs = buffer_differences(sim_a, sim_b)
    assert not diffs, "signals differ (name, elements, largest difference, first index): %s" % diffs
