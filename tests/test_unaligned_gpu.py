"""The `_unaligned` pipelined kernels against the oracle: every kernel by name, every combination of
odd and even Q/K/V slices at tile edges, with infinities and NaNs in everything around the slices
(a neighbouring element that reached a product would show), the routes through the selection, and
the exactness of sharply peaked rows."""

import dataclasses
import itertools
import math
import os
import re

import numpy as np
import pytest

import flashcheck as fc
import notcute_flash as nc
from flash_workloads import Workload

pytestmark = pytest.mark.gpu

POISON = {"f16": np.array([0x7C00, 0x7E00, 0xFC00], np.uint16), "bf16": np.array([0x7F80, 0x7FC0, 0xFF80], np.uint16)}


def poisoned(wl: Workload, arr, which, offset):
    """The tensor in a buffer `offset` elements longer, all that is not an active element poisoned."""
    out = np.resize(POISON[wl.dtype], arr.size + offset + 8)
    b = np.arange(wl.batch_heads)[:, None, None] * wl.stride(which)
    idx = (b + np.arange(wl.seq_len)[None, :, None] * wl.row(which) + np.arange(wl.head_dim)).reshape(-1)
    out[idx + offset] = arr[idx]
    return out


def check(gpu, wl, offs, name=None):
    print(f"[case] {wl.describe()} {wl.dtype} offsets={offs} {name or ''}", flush=True)
    tensors = wl.make_inputs()
    o_init = np.full(wl.length("o"), fc.SENTINEL, dtype=np.float32)
    ref = fc.oracle(wl, *tensors, o_init=o_init)
    bufs = [nc.DeviceBuffer.from_array(poisoned(wl, t, w, f)) for t, w, f in zip(tensors, "qkv", offs)]
    bufs.append(nc.DeviceBuffer.from_array(o_init))
    try:
        ptr = [b.ptr + 2 * f for b, f in zip(bufs, offs)] + [bufs[3].ptr]
        sel = nc.select_kernel_for(wl.options(), *ptr)
        if name is None:
            name, grid, threads = sel.name.decode(), tuple(sel.grid), sel.threads
        else:
            m = re.search(r"_q(\d+)s(\d+)p", name)
            sel = nc.KernelSelection()
            sel.block_m, threads = 32 * int(m.group(1)), 64 * int(m.group(1)) * int(m.group(2))
            grid = (-(-wl.seq_len // sel.block_m) * wl.batch_heads,)
        args = nc.pack_args(wl.options(), sel, *ptr)
        gpu.get_function(name).launch(grid, (threads,), nc.kernel_params(name, args))
        nc.synchronize()
        out = bufs[3].download(np.float32, wl.length("o"))
    finally:
        for b in bufs:
            b.free()
    # the parity bar of the element type (f16 2e-3 / 1e-2, bf16 8e-3 / 4e-2): the same arithmetic as the
    # aligned kernels, in another order over the head columns
    max_abs, max_rel = fc.parity_bar(wl.dtype)
    fc.assert_parity(out, ref, fc.active_index(wl), name, max_abs=max_abs, max_rel=max_rel)
    fc.assert_pads_untouched(out, o_init, wl, name)
    return name


def _names():
    src = open(os.path.join(os.path.dirname(__file__), "..", "not-cute-zig_amd", "csrc", "flash_fwd.hip")).read()
    names = re.findall(r"NC_FLASH_UNALIGNED_PIPE_KERNEL\((nc_flash_fwd_\w+),", src)
    return sorted(n + t for n in names for t in ("", "_bf16"))


@pytest.mark.parametrize("name", _names())
def test_each_unaligned_kernel(gpu, name):
    """S = 1100: several blocks per wave in every kernel, no multiple of any tile. Three slices whose
    strides make Q, K, V even and odd in turn; no kernel may use scratch."""
    d = int(re.search(r"_d(\d+)_", name).group(1))
    assert gpu.get_function(name).attributes().local_size_bytes == 0
    s = 1100
    wl = Workload(f"un_{name}", 3, s, d, "_causal" in name, 1.0 / math.sqrt(d), (("normal", 0.0, 1.0),) * 3, seed=31,
                  q_stride=s * d + 17, k_stride=s * d + 19, v_stride=s * d + 23, o_stride=s * d + 29,
                  dtype="bf16" if name.endswith("_bf16") else "f16")
    check(gpu, wl, (0, 1, 0), name)


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("causal", [False, True])
def test_phases_and_lengths(gpu, d, causal):
    """Every combination of odd and even Q, K, V at the lengths around the tiles and blocks, packed and
    padded rows (an odd Q pitch among them)."""
    for i, s in enumerate((1, 2, 31, 32, 33, 64, 65, 127, 128, 129, 257, 513)):
        row = {} if i % 3 else dict(q_row=d + 5, k_row=d + 6, v_row=d + 6, o_row=d + 3)
        for offs in itertools.product((0, 1), repeat=3):
            wl = Workload(f"ph{s}", 2, s, d, causal, (-0.3 if i % 4 == 3 else 1.0 / math.sqrt(d)),
                          (("normal", 0.0, 1.0),) * 3, seed=40 + i, o_stride=s * (d + 3) + 1, **row)
            check(gpu, wl, offs)


@pytest.mark.parametrize("bh,s,d,causal", [(8, 250, 32, True), (96, 333, 64, True), (24, 1500, 64, False),
                                           (128, 700, 16, False), (3, 3100, 64, True), (96, 130, 32, False)])
@pytest.mark.parametrize("offs", [(2, 4, 6), (1, 2, 4), (0, 3, 0), (0, 0, 5)])
def test_dispatched_routes(gpu, bh, s, d, causal, offs):
    """Through the selection (causal BH=3 S=3100 would take the pair split if it were 16-byte aligned)."""
    wl = Workload(f"route_{bh}_{s}_{d}", bh, s, d, causal, 1.0 / math.sqrt(d), (("normal", 0.0, 1.0),) * 3, seed=50)
    opts = wl.options()
    sel = nc.select_kernel_for(opts, *[(1 << 20) + 2 * f for f in offs], 1 << 20)
    assert sel.name.decode().endswith("_unaligned")
    assert sel.scratch_bytes == 0
    check(gpu, wl, offs)


@pytest.mark.parametrize("bh,s,d,causal", [(16, 2048, 64, True), (96, 333, 64, False), (8, 1024, 64, True),
                                           (128, 1000, 32, True), (64, 1500, 16, False)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_peaked_rows_are_as_exact_as_the_generic_kernels(gpu, bh, s, d, causal, dtype):
    """Logits of sigma 3, where one key can hold most of a row: its weight is exactly 1 only where the
    running max follows every tile. The error against float64 has to be no larger than the generic
    kernel's, which takes the max per tile. Both errors are maxima over ~1e5 independent roundings of
    the weights (2^-11 or 2^-8 relative) and the factor covers their spread: a lazy max is at 1.5 to 2.
    Both stand for themselves too: each meets the oracle within the parity bar, and their rms error stays
    below u / sqrt(3) (a weight's rounding, u = 2^-11 or 2^-8 at most) * 1/2 (the largest share of a weight
    that is not the row's largest) * sqrt(2) (rms of v - o), 2.0e-4 and 1.6e-3."""
    wl = Workload(f"peak_{bh}_{s}_{d}", bh, s, d, causal, 1.0 / math.sqrt(d),
                  (("normal", 0.0, 3 ** 0.5),) * 2 + (("normal", 0.0, 1.0),), seed=60, q_stride=s * d + 17, dtype=dtype)
    tensors = wl.make_inputs()
    rows = np.arange(0, s, max(1, s // 64))
    ref = fc.oracle(wl, *tensors, rows=rows)
    idx = fc.active_index(wl, rows)
    odd = dataclasses.replace(wl, k_row=d + 1, v_row=d + 1, k_stride=0, v_stride=0)
    errs = {}
    o_init = np.full(wl.length("o"), fc.SENTINEL, np.float32)
    max_abs, max_rel = fc.parity_bar(dtype)
    bufs = [nc.DeviceBuffer.from_array(t) for t in (*tensors, o_init)]
    try:
        ptr = [b.ptr for b in bufs]
        for kind, opts in (("generic", odd.options()), ("unaligned", wl.options())):
            sel = nc.select_kernel_for(opts, *ptr)
            name = sel.name.decode()
            print(f"[case] {wl.describe()} {dtype} {name}", flush=True)
            assert ("_m64_" in name) == (kind == "generic")
            bufs[3].upload(o_init)
            args = nc.pack_args(wl.options(), sel, *ptr)
            gpu.get_function(name).launch(tuple(sel.grid), (sel.threads,), nc.kernel_params(name, args))
            nc.synchronize()
            out = bufs[3].download(np.float32, wl.length("o"))
            fc.assert_parity(out, ref, idx, name, max_abs=max_abs, max_rel=max_rel)
            err = np.abs(out[idx].astype(np.float64) - ref[idx])
            errs[kind] = (float(err.max()), float((err ** 2).mean() ** 0.5))
    finally:
        for b in bufs:
            b.free()
    print(f"[ok] {errs}", flush=True)
    assert max(e[1] for e in errs.values()) <= (1.6e-3 if dtype == "bf16" else 2.0e-4)
    assert errs["unaligned"][0] <= 1.25 * errs["generic"][0]
    assert errs["unaligned"][1] <= 1.05 * errs["generic"][1]


@pytest.mark.parametrize("bh,s,d,causal", [(16, 1500, 64, False), (32, 700, 64, True), (8, 250, 32, True),
                                           (96, 520, 32, False), (64, 1100, 16, True), (4, 1979, 64, False)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_output_is_the_generic_kernels(gpu, bh, s, d, causal, dtype):
    """Both round a weight at the same running max, so they differ only where an exponent's f32 rounding
    (of |scores| up to 8: four units of 2^-21) takes a weight across the middle between two neighbours,
    2^-11 or more apart (f16): at most a share 2 * 4 * 2^-21 * ln 2 / 2^-11 of the weights, by sqrt(12)
    times the rms rounding error each. That is sqrt(12 * 0.0054) = 0.25 of the error against float64;
    0.3 with the sums' own rounding. Weights rounded at other maxima differ by 0.8 of it and more."""
    wl = Workload(f"same_{bh}_{s}_{d}", bh, s, d, causal, 1.0 / math.sqrt(d), (("normal", 0.0, 1.0),) * 3, seed=70,
                  q_stride=s * d + 17, k_stride=s * d + 19, v_stride=s * d + 23, o_stride=s * d + 29, dtype=dtype)
    tensors = wl.make_inputs()
    rows = np.arange(0, s, max(1, s // 64))
    idx = fc.active_index(wl, rows)
    full = fc.oracle(wl, *tensors, rows=rows)
    ref = full[idx].astype(np.float64)
    max_abs, max_rel = fc.parity_bar(dtype)
    odd = dataclasses.replace(wl, k_row=d + 1, v_row=d + 1, k_stride=0, v_stride=0)
    o_init = np.full(wl.length("o"), fc.SENTINEL, np.float32)
    bufs = [nc.DeviceBuffer.from_array(t) for t in (*tensors, o_init)]
    out = {}
    try:
        ptr = [b.ptr for b in bufs]
        for kind, opts in (("generic", odd.options()), ("unaligned", wl.options())):
            sel = nc.select_kernel_for(opts, *ptr)
            name = sel.name.decode()
            print(f"[case] {wl.describe()} {dtype} {name}", flush=True)
            assert ("_m64_" in name) == (kind == "generic")
            bufs[3].upload(o_init)
            args = nc.pack_args(wl.options(), sel, *ptr)
            gpu.get_function(name).launch(tuple(sel.grid), (sel.threads,), nc.kernel_params(name, args))
            nc.synchronize()
            o = bufs[3].download(np.float32, wl.length("o"))
            fc.assert_parity(o, full, idx, name, max_abs=max_abs, max_rel=max_rel)
            out[kind] = o[idx].astype(np.float64)
    finally:
        for b in bufs:
            b.free()
    err = np.linalg.norm(out["generic"] - ref)
    diff = np.linalg.norm(out["unaligned"] - out["generic"])
    print(f"[ok] difference {diff / np.linalg.norm(ref):.2e} error {err / np.linalg.norm(ref):.2e}", flush=True)
    assert diff <= 0.3 * err
