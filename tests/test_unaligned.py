"""Dispatch of slices that are not 16-byte aligned (no GPU): the `_unaligned` pipelined kernels take
every layout at elements with one even row stride for K and V, the generic kernels the rest."""

import itertools

import pytest

import notcute_flash as nc

BASE = 1 << 20


def route(bh, s, d, causal, q=BASE, k=BASE, v=BASE, o=BASE, rows=(0, 0, 0, 0), pads=(0, 0, 0, 0), dtype="f16"):
    r = [x or d for x in rows]
    opts = nc.options(batch_heads=bh, seq_len=s, head_dim=d, causal=causal, dtype=dtype, q_row_stride=rows[0],
                      k_row_stride=rows[1], v_row_stride=rows[2], o_row_stride=rows[3], q_stride=s * r[0] + pads[0],
                      k_stride=s * r[1] + pads[1], v_stride=s * r[2] + pads[2], o_stride=s * r[3] + pads[3])
    sel = nc.select_kernel_for(opts, q, k, v, o)
    name = sel.name.decode()
    family = "generic" if "_m64_" in name else "unaligned" if "_unaligned" in name else "pipe"
    return family, sel


SHAPES = [(1, 1, 16), (3, 49, 16), (8, 250, 32), (8, 1024, 64), (16, 1500, 64), (64, 2048, 16), (128, 1000, 32),
          (64, 512, 64), (4, 8192, 64), (32, 4096, 64)]


@pytest.mark.parametrize("bh,s,d", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
def test_route_follows_the_layout(bh, s, d, causal):
    for offs in itertools.product((0, 1, 2, 4), repeat=3):  # elements past 16-byte alignment of Q, K, V
        ptr = dict(zip("qkv", (BASE + 2 * x for x in offs)))
        family, sel = route(bh, s, d, causal, **ptr)
        assert family == ("unaligned" if any(offs) else "pipe"), offs
        assert sel.aligned == (1 if not any(offs) else 0)
    for pads in itertools.product((0, 3, 6), repeat=3):
        family, sel = route(bh, s, d, causal, pads=pads + (5,))
        assert family == "unaligned", pads  # (the float padding of O alone is enough)
        assert sel.aligned == 0
    # O: any float; an address between floats, and odd, differing or odd-element K/V rows: generic
    assert route(bh, s, d, causal, o=BASE + 4)[0] == "unaligned"
    assert route(bh, s, d, causal, o=BASE + 2)[0] == "generic"
    assert route(bh, s, d, causal, q=BASE + 1)[0] == "generic"
    assert route(bh, s, d, causal, rows=(d + 2, d + 2, d + 4, d + 1))[0] == "generic"
    assert route(bh, s, d, causal, rows=(d + 1, d + 2, d + 2, 0))[0] == "unaligned"
    assert route(bh, s, d, causal, k=BASE + 2, rows=(0, d + 2, d + 4, 0))[0] == "generic"
    assert route(bh, s, d, causal, rows=(0, d + 1, d + 1, 0))[0] == "generic"


@pytest.mark.parametrize("bh,s,d", SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_unaligned_selection_is_launchable(bh, s, d, dtype):
    for causal in (False, True):
        # an odd K/V row stride: the generic kernel
        _, gen = route(bh, s, d, causal, rows=(0, d + 1, d + 1, 0), dtype=dtype)
        _, un = route(bh, s, d, causal, k=BASE + 2, dtype=dtype)
        assert un.name.decode().endswith("_unaligned_bf16" if dtype == "bf16" else "_unaligned")
        # (threads per row: 2 per key split) no fewer splits than the generic kernel, since a row's
        # exactness grows with them
        assert un.threads // un.block_m >= gen.threads // gen.block_m and un.scratch_bytes == 0
        assert un.grid[0] == -(-s // un.block_m) * bh and un.grid[1] == un.grid[2] == 1


def test_no_new_scratch_and_no_new_refusals():
    """The pair split's scratch stays with 16-byte aligned slices; a grid that only the generic
    kernels' workgroups fit keeps them."""
    assert route(1, 4096, 64, True)[1].scratch_bytes > 0
    for ptr in (BASE + 4, BASE + 2):
        assert route(1, 4096, 64, True, q=ptr)[1].scratch_bytes == 0
    for d in (16, 32, 64):
        for ptr in (BASE + 4, BASE + 2):
            family, sel = route((1 << 23) - 1, 1, d, False, q=ptr)
            assert sel.grid[0] * sel.threads <= 0xFFFFFFFF
    assert route((1 << 24) - 1, 1, 32, False, q=BASE + 2)[1].threads == 256


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("causal", [False, True])
def test_key_splits_are_the_generic_kernels(d, causal):
    """A weight is rounded at the running max of its key split, so a call's output stays what the generic
    kernel gives it only with that kernel's number of splits."""
    for bh in (1, 3, 8, 16, 24, 64, 100, 192, 500):
        for s in (1, 32, 33, 129, 250, 333, 700, 1500, 2048, 4096, 8192):
            gen = route(bh, s, d, causal, rows=(0, d + 1, d + 1, 0))[1]
            for ptr in (BASE + 2, BASE + 4):
                assert route(bh, s, d, causal, k=ptr)[1].kv_splits == gen.kv_splits, (bh, s)


@pytest.mark.parametrize("bh,s,d,causal,odd,dword", [
    # K and V of an XCD's slices against its L2 (d = 64, the 128-row generic kernel otherwise)
    (64, 4000, 64, False, "unaligned", "unaligned"), (199, 2048, 64, False, "generic", "generic"),
    (199, 2048, 64, True, "generic", "generic"), (100, 4000, 64, False, "generic", "generic"),
    (100, 4000, 64, True, "unaligned", "unaligned"), (333, 4000, 64, True, "generic", "generic"),
    (4095, 512, 64, False, "generic", "generic"), (1023, 256, 64, False, "unaligned", "generic"),
    (64, 8192, 64, True, "unaligned", "unaligned"), (5387, 368, 64, False, "unaligned", "generic"),
    # few reads of K and V
    (1000, 64, 64, False, "unaligned", "unaligned"), (495, 79, 64, True, "unaligned", "generic"),
    # one or two tiles per wave (the 64-row generic kernel)
    (229, 43, 64, False, "unaligned", "generic"), (820, 18, 16, False, "generic", "generic"),
    (920, 65, 32, True, "unaligned", "generic"), (920, 129, 32, True, "unaligned", "unaligned"),
    # eight key splits: always
    (8, 20, 16, True, "unaligned", "unaligned"), (3, 8192, 64, True, "unaligned", "unaligned")])
def test_generic_kernels_where_they_are_faster(bh, s, d, causal, odd, dword):
    assert route(bh, s, d, causal, pads=(17, 19, 23, 29))[0] == odd
    assert route(bh, s, d, causal, q=BASE + 2)[0] == odd
    assert route(bh, s, d, causal, pads=(2, 6, 10, 3))[0] == dword
    assert route(bh, s, d, causal, o=BASE + 4)[0] == dword


def test_dispatch_holds_at_the_largest_sizes():
    """No overflow in the rule: the largest counts still select a kernel or are refused for their grid."""
    for bh, s in ((1, (1 << 31) - 257), ((1 << 32) - 1, 1), ((1 << 32) - 1, 200), (1 << 31, 70), (7, 1 << 23)):
        for d in (16, 64):
            try:
                sel = route(bh, s, d, False, q=BASE + 2)[1]
            except nc.NcError:
                continue
            assert sel.grid[0] * sel.threads <= 0xFFFFFFFF
