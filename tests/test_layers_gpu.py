"""The launch order of the causal pipelined kernels (alternate layers of workgroups turned round): every
query block of every head is computed exactly once, whatever the head count, at the edges of the layers."""

import math

import numpy as np
import pytest

import flashcheck as fc
import notcute_flash as nc
from flash_workloads import Workload

pytestmark = pytest.mark.gpu

# (kernel, rows per workgroup, threads)
KERNELS = [("d64_q8s1p2t2", 256, 512), ("d64_q4s1p2t2", 128, 256), ("d64_q2s4p2", 64, 512), ("d64_q1s8p1", 32, 512),
           ("d32_q4s1p3", 128, 256), ("d16_q4s1p2t2", 128, 256), ("d32_q1s8p2", 32, 512),
           ("d64_q2s2p2_u", 64, 256)]


@pytest.mark.parametrize("kernel,bm,threads", KERNELS)
@pytest.mark.parametrize("bh,blocks", [(1, 3), (2, 129), (3, 86), (4, 65), (8, 32), (8, 33), (8, 65), (12, 43), (24, 21),
                                       (40, 13), (64, 5), (256, 2), (257, 2), (5, 103), (1, 1), (8, 1), (257, 1),
                                       (1000, 1), (1027, 1), (8, 2), (300, 2), (94, 7)])
def test_every_block_once(gpu, kernel, bm, threads, bh, blocks):
    """V constant 1 per (head, column) pattern makes O = V whatever the scores, so each row shows whether
    it was written, from its own head; a sentinel shows rows that were not. Grids of just under, at and
    just over one and two layers of 256 workgroups, and one or two blocks per head."""
    d, s = int(kernel[1:3]), blocks * bm - 7
    un = kernel.endswith("_u")
    wl = Workload(f"layers_{kernel}", bh, s, d, True, 1.0 / math.sqrt(d), (("uniform", -1.0, 1.0),) * 3, seed=81)
    if un:
        wl.k_stride = wl.v_stride = s * d + 1
    n = wl.length("q")
    q = np.resize(nc.fill_uniform(4096, 5, 0), n)
    k = np.resize(nc.fill_uniform(4099, 5, 1), wl.length("k"))
    head = (np.arange(bh) % 61 + 1).astype(np.float16).view(np.uint16)
    v = np.zeros(wl.length("v"), np.uint16)
    for b in range(bh):
        v[b * wl.stride("v"): b * wl.stride("v") + s * d] = head[b]
    o_init = np.full(n, fc.SENTINEL, dtype=np.float32)
    name = f"nc_flash_fwd_{kernel.replace('_u', '')}_causal" + ("_unaligned" if un else "")
    print(f"[case] {name} BH={bh} S={s} workgroups={bh * blocks}", flush=True)
    bufs = [nc.DeviceBuffer.from_array(x) for x in (q, k, v, o_init)]
    try:
        sel = nc.KernelSelection()
        sel.block_m = bm
        args = nc.pack_args(wl.options(), sel, *[b.ptr for b in bufs])
        gpu.get_function(name).launch((bh * blocks,), (threads,), [args])
        nc.synchronize()
        out = bufs[3].download(np.float32, n).reshape(bh, s, d)
    finally:
        for b in bufs:
            b.free()
    # O = sum(w v) / sum(w) with v constant and the same rounded w in both sums: f32 rounding only
    want = (np.arange(bh) % 61 + 1).astype(np.float32)[:, None, None]
    assert np.max(np.abs(out / want - 1.0)) <= 1e-4


# Workgroups per CU that the launch order of each causal shared-staging kernel assumes (pipe_layers)
LAYERS = {"d64_q8s1p2t2": 2, "d64_q4s1p2t2": 4, "d64_q2s4p2": 2, "d64_q2s2p2_u": 3, "d32_q4s1p3": 5, "d32_q2s4p2": 2,
          "d32_q2s2p2_u": 6, "d16_q4s1p2t2": 6, "d16_q2s4p2": 3, "d16_q2s2p2_u": 7}


@pytest.mark.parametrize("dtype", ["", "_bf16"])
@pytest.mark.parametrize("kernel", sorted(LAYERS))
def test_layers_are_the_occupancy(gpu, kernel, dtype):
    q, s = (int(kernel[kernel.index(c) + 1]) for c in "qs")
    name = f"nc_flash_fwd_{kernel.replace('_u', '')}_causal" + ("_unaligned" if "_u" in kernel else "") + dtype
    assert gpu.get_function(name).max_active_blocks(64 * q * s) == LAYERS[kernel]
