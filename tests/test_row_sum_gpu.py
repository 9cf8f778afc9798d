"""The row sum on the matrix cores mixes queries n and n + 16 of a 32-query tile in one MFMA column. A
NaN or an overflowing weight of one must not reach the other: kernels of every geometry, launched by
name (the packed-slice forms, the `_unaligned` kernels and the reference-named symbol that run the same
body among them), with a NaN query, with rows whose scores keep growing (the running max moves at every
tile), and with rows that see no key until late."""

import ctypes
import math
import re

import numpy as np
import pytest

import flashcheck as fc
import notcute_flash as nc
from flash_workloads import Workload

pytestmark = pytest.mark.gpu

KERNELS = ["d64_q8s1p2t2", "d64_q4s1p2t2", "d64_q2s4p2", "d64_q1s8p2", "d32_q4s1p3", "d32_q2s4p2", "d32_q1s8p1",
           "d16_q4s1p2t2", "d16_q2s4p2", "d16_q1s8p2", "d16_q1s8p1", "d16_q1s8p2d", "d16_q1s8p1d",
           "d64_q2s2p2_u", "d32_q2s2p2_u", "d16_q2s2p2_u", "d64_q1s8p1_u", "d16_q1s8p2_u"]


def launch(gpu, wl, name, tensors):
    o_init = np.full(wl.length("o"), fc.SENTINEL, dtype=np.float32)
    bufs = [nc.DeviceBuffer.from_array(x) for x in (*tensors, o_init)]
    try:
        m = re.search(r"_q(\d+)s(\d+)p", name)
        sel = nc.KernelSelection()
        sel.block_m, threads = 32 * int(m.group(1)), 64 * int(m.group(1)) * int(m.group(2))
        args = nc.pack_args(wl.options(), sel, *[b.ptr for b in bufs])
        blocks = -(-wl.seq_len // sel.block_m)
        grid = (wl.batch_heads, 1, blocks) if re.search(r"p\d+d_", name) else (blocks * wl.batch_heads,)
        gpu.get_function(name).launch(grid, (threads,), nc.kernel_params(name, args))
        nc.synchronize()
        return bufs[3].download(np.float32, wl.length("o"))
    finally:
        for b in bufs:
            b.free()


def rows_workload(d, causal, dtype):
    """Workload, inputs, the oracle's output and the rows of slice 1 whose query holds a NaN."""
    wl = Workload(f"rows_d{d}", 2, 700, d, causal, 1.0 / math.sqrt(d), (("normal", 0.0, 1.0),) * 3, seed=71, dtype=dtype)
    q, k, v = wl.make_inputs()
    nan_bits = np.uint16(0x7E00 if dtype == "f16" else 0x7FC0)
    k2 = k.reshape(2, 700, d).copy()
    q2 = q.reshape(2, 700, d).copy()
    # slice 0: column 0 of K grows with the key, column 0 of Q is large in every 16th + 3 row: those rows'
    # scores rise by many powers of two from tile to tile, and only theirs
    def enc(x):
        x = np.asarray(x, np.float32)
        return x.astype(np.float16).view(np.uint16) if dtype == "f16" else (x.view(np.uint32) >> 16).astype(np.uint16)

    k2[0, :, 0] = enc(np.arange(700) / 32.0)
    q2[0, :, 0] = 0
    q2[0, 3::16, 0] = enc(np.full(len(range(3, 700, 16)), 8.0))
    nan_rows = [5, 16, 37, 250, 511, 699]  # slice 1
    q_clean = q2.copy()
    for r in nan_rows:
        q2[1, r, 1] = nan_bits
    o_init = np.full(wl.length("o"), fc.SENTINEL, dtype=np.float32)
    ref = fc.oracle(wl, q_clean.reshape(-1), k2.reshape(-1), v, o_init=o_init).reshape(2, 700, d)
    return wl, (q2.reshape(-1), k2.reshape(-1), v), ref, nan_rows


def check_rows(out, ref, nan_rows, dtype, name):
    assert np.all(np.isnan(out[1, nan_rows])), "a NaN query gives NaN"
    keep = np.ones((2, 700), bool)
    keep[1, nan_rows] = False
    assert np.all(np.isfinite(out[keep])), "and no other row does"
    # the parity bar of the element type, on every other row
    max_abs, max_rel = fc.parity_bar(dtype)
    fc.assert_parity(out[keep].reshape(-1), ref[keep].reshape(-1), np.arange(out[keep].size), name, max_abs=max_abs,
                     max_rel=max_rel)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kernel", KERNELS)
def test_rows_stay_apart(gpu, kernel, causal, dtype):
    d = int(kernel[1:3])
    wl, tensors, ref, nan_rows = rows_workload(d, causal, dtype)
    suffix = ("_unaligned" if kernel.endswith("_u") else "") + ("_bf16" if dtype == "bf16" else "")
    name = f"nc_flash_fwd_{kernel.replace('_u', '')}_{'causal' if causal else 'full'}{suffix}"
    print(f"[case] {name}", flush=True)
    check_rows(launch(gpu, wl, name, tensors).reshape(2, 700, d), ref, nan_rows, dtype, name)


@pytest.mark.parametrize("name", ["flash_attention_fwd_v2", "flash_attention_fwd_h64_bn32"])
@pytest.mark.parametrize("causal", [False, True])
def test_rows_stay_apart_in_the_reference_named_symbols(gpu, name, causal):
    """From 16384 workgroups these run the same body, 64 rows on two query waves: 374 slices (187 times
    the same two) of 44 16-row blocks. Every copy has the same bits."""
    wl, tensors, ref, nan_rows = rows_workload(64, causal, "f16")
    n, copies = wl.stride("q"), 187
    print(f"[case] {name} causal={causal}", flush=True)
    bufs = [nc.DeviceBuffer.from_array(np.tile(t, copies)) for t in tensors]
    bufs.append(nc.DeviceBuffer.from_array(np.full(2 * copies * n, fc.SENTINEL, np.float32)))
    try:
        params = [ctypes.c_void_p(b.ptr) for b in bufs] + [ctypes.c_uint64(x) for x in (700, 64, n, n, n, n)]
        params += [ctypes.c_float(wl.scale), ctypes.c_uint32(causal)]
        gpu.get_function(name).launch((44, 2 * copies), (128,), params)
        nc.synchronize()
        out = bufs[3].download(np.float32, 2 * copies * n).reshape(copies, 2, 700, 64)
    finally:
        for b in bufs:
            b.free()
    check_rows(out[0], ref, nan_rows, "f16", name)
    assert np.all(out.view(np.uint32) == out[:1].view(np.uint32))
