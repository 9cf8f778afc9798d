"""The row sum on the matrix cores mixes queries n and n + 16 of a 32-query tile in one MFMA column. A
NaN or an overflowing weight of one must not reach the other: kernels of every geometry, launched by
name, with a NaN query, with rows whose scores keep growing (the running max moves at every tile), and
with rows that see no key until late."""

import math
import re

import numpy as np
import pytest

import flashcheck as fc
import notcute_flash as nc
from flash_workloads import Workload

pytestmark = pytest.mark.gpu

KERNELS = ["d64_q8s1p2t2", "d64_q4s1p2t2", "d64_q2s4p2", "d64_q1s8p2", "d32_q4s1p3", "d32_q2s4p2", "d32_q1s8p1",
           "d16_q4s1p2t2", "d16_q2s4p2", "d16_q1s8p2", "d16_q1s8p1"]


def launch(gpu, wl, name, tensors):
    o_init = np.full(wl.length("o"), fc.SENTINEL, dtype=np.float32)
    bufs = [nc.DeviceBuffer.from_array(x) for x in (*tensors, o_init)]
    try:
        m = re.search(r"_q(\d+)s(\d+)p", name)
        sel = nc.KernelSelection()
        sel.block_m, threads = 32 * int(m.group(1)), 64 * int(m.group(1)) * int(m.group(2))
        args = nc.pack_args(wl.options(), sel, *[b.ptr for b in bufs])
        gpu.get_function(name).launch((-(-wl.seq_len // sel.block_m) * wl.batch_heads,), (threads,), [args])
        nc.synchronize()
        return bufs[3].download(np.float32, wl.length("o"))
    finally:
        for b in bufs:
            b.free()


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kernel", KERNELS)
def test_rows_stay_apart(gpu, kernel, causal, dtype):
    d = int(kernel[1:3])
    wl = Workload(f"rows_{kernel}", 2, 700, d, causal, 1.0 / math.sqrt(d), (("normal", 0.0, 1.0),) * 3, seed=71, dtype=dtype)
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
    suffix = "_bf16" if dtype == "bf16" else ""
    name = f"nc_flash_fwd_{kernel}_{'causal' if causal else 'full'}{suffix}"
    print(f"[case] {name}", flush=True)
    out = launch(gpu, wl, name, (q2.reshape(-1), k2.reshape(-1), v)).reshape(2, 700, d)
    assert np.all(np.isnan(out[1, nan_rows])), "a NaN query gives NaN"
    keep = np.ones((2, 700), bool)
    keep[1, nan_rows] = False
    assert np.all(np.isfinite(out[keep])), "and no other row does"
    # the parity bar of the element type, on every other row
    max_abs, max_rel = fc.parity_bar(dtype)
    fc.assert_parity(out[keep].reshape(-1), ref[keep].reshape(-1), np.arange(keep.sum() * d), name, max_abs=max_abs,
                     max_rel=max_rel)
