"""Performance cases of the flash-attention forward: what a program that uses this library has it
compute, through the public Python entry points (flash_launch, and HIP graphs of such launches).

A case is one call, or the calls of a stack of layers: made one by one, or captured once into a HIP
graph and replayed (the way short launches are issued when latency matters):
  batch_heads, seq_len, head_dim, causal, dtype ("f16" | "bf16")
  layout   "dense"  packed slices
           "rows"   every row padded by 8 elements (16-byte aligned rows)
           "odd"    slices padded by 17/19/23/29 elements (Q/K/V/O), as the reference's smoke cases pad
                    theirs: slice bases have no common alignment beyond the element's own
  sigma    standard deviation of Q and K (1: ordinary logits; 3: sharp ones, where few keys dominate)
  layers   calls of one pass, each on tensors of its own
  graph    the calls are a captured graph, replayed once a pass
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "not-cute-zig_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import notcute_flash as nc  # noqa: E402

LAYERS = 12
ROW_PAD = 8
ODD_PADS = (17, 19, 23, 29)
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


def _case(name, batch_heads, seq_len, head_dim, causal, dtype="f16", layout="dense", sigma=1.0, layers=1,
          graph=False):
    return {"name": name, "batch_heads": batch_heads, "seq_len": seq_len, "head_dim": head_dim, "causal": causal,
            "dtype": dtype, "layout": layout, "sigma": sigma, "layers": layers, "graph": graph}


def listed():
    return [
        # The smallest calls (a 32-token prompt, one head), made one by one through a stack of layers:
        # the cost of a call itself.
        _case("calls_tiny", 1, 32, 16, False, layers=LAYERS),
        # A short prompt through a captured stack of layers, rows padded to a pitch of 40.
        _case("stack_short_rows", 8, 128, 32, True, layout="rows", layers=LAYERS, graph=True),
        # The same kind of stack on slices with the reference's odd pads, ragged length.
        _case("stack_short_odd", 8, 250, 32, True, layout="odd", layers=LAYERS, graph=True),
        # The headline shape: a 1024-token causal prefill of 8 heads, as a captured stack.
        _case("stack_headline", 8, 1024, 64, True, layers=LAYERS, graph=True),
        # Many short ragged sequences in a batch (192 heads x 333 tokens), bf16.
        _case("batch_ragged_bf16", 192, 333, 64, True, dtype="bf16"),
        # An encoder-style full attention at a mid size on odd slices.
        _case("encoder_odd", 16, 1500, 64, False, layout="odd"),
        # Small heads over mid-length sequences: full attention at head_dim 16 ...
        _case("heads16_full", 64, 2048, 16, False),
        # ... and causal at head_dim 32, one short of a tile multiple.
        _case("heads32_causal", 64, 2047, 32, True),
        # A long prompt over few heads (one sequence on a sharded model): little parallelism over heads.
        _case("long_few_heads", 4, 8192, 64, True),
        # A long causal prefill in bf16 with padded rows, ragged length.
        _case("long_rows_bf16", 32, 4000, 64, True, dtype="bf16", layout="rows"),
        # Large full attention (32 heads x 4096).
        _case("large_full", 32, 4096, 64, False),
        # The largest: a long causal prefill over 64 heads with sharp logits.
        _case("largest_causal", 64, 8192, 64, True, sigma=3.0),
    ]


def draw(rng):
    head_dim = rng.choice((64, 64, 64, 32, 32, 16))
    causal = rng.random() < 0.6
    dtype = "bf16" if rng.random() < 0.3 else "f16"
    layout = rng.choice(("dense", "dense", "dense", "rows", "odd", "odd"))
    seq_len = int(round(math.exp(rng.uniform(math.log(32), math.log(8192)))))
    if rng.random() < 0.3:
        seq_len = max(32, seq_len // 64 * 64)  # lengths that are tile multiples are common too
    batch_heads = int(round(math.exp(rng.uniform(0.0, math.log(256)))))
    # (query, key) pairs of one call: at most those of the largest listed case, and a quarter of them
    # at the head sizes and layouts whose pairs cost more time per flop
    most = 64 * 8192 * 8192 // 2
    if layout == "odd" or head_dim < 64:
        most //= 4
    pairs = seq_len * seq_len // (2 if causal else 1)
    batch_heads = max(1, min(batch_heads, most // pairs))
    short = batch_heads * pairs <= 8 * 1024 * 1024
    case = _case("", batch_heads, seq_len, head_dim, causal, dtype, layout, rng.choice((1.0, 1.0, 3.0)),
                 LAYERS if short else 1, short and rng.random() < 0.75)
    del case["name"]
    return case


_session = None


def _context():
    """The process's module and graph stream, made once as a program does at start-up."""
    global _session
    if _session is None:
        torch.cuda.init()
        nc.init()
        _session = (nc.Module.load_embedded(), nc.Stream())
    return _session


class _Buffer:
    """A torch tensor as the buffer object flash_launch takes (device address and size)."""

    def __init__(self, tensor):
        self.ptr = tensor.data_ptr()
        self.nbytes = tensor.numel() * tensor.element_size()


class _Stack:
    """A captured graph of launches, released with the state that holds it."""

    def __init__(self, stream, body):
        self.stream = stream
        self.graph = nc.Graph.capture(stream, body)

    def __call__(self):
        self.graph.launch(self.stream)

    def __del__(self):
        self.graph.destroy()


def _strides(case):
    """(row pitch, the four slice strides Q/K/V/O) in elements."""
    row = case["head_dim"] + (ROW_PAD if case["layout"] == "rows" else 0)
    pads = ODD_PADS if case["layout"] == "odd" else (0, 0, 0, 0)
    return row, tuple(case["seq_len"] * row + p for p in pads)


def _inputs(case, seed):
    """Q, K, V as [calls, batch_heads * slice stride] tensors, paddings filled like the rest."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    calls = case["layers"]
    _, strides = _strides(case)
    out = []
    for which, stride in zip("qkv", strides):
        x = torch.randn(calls, case["batch_heads"] * stride, generator=gen, device="cuda", dtype=torch.float32)
        out.append((x * (case["sigma"] if which != "v" else 1.0)).to(DTYPES[case["dtype"]]))
    return out


def prepare(case, seed):
    module, stream = _context()
    q, k, v = _inputs(case, seed)
    row, strides = _strides(case)
    calls = case["layers"]
    o = torch.zeros(calls, case["batch_heads"] * strides[3], device="cuda", dtype=torch.float32)
    opts = nc.options(batch_heads=case["batch_heads"], seq_len=case["seq_len"], head_dim=case["head_dim"],
                      q_stride=strides[0], k_stride=strides[1], v_stride=strides[2], o_stride=strides[3],
                      causal=case["causal"], q_row_stride=row, k_row_stride=row, v_row_stride=row, o_row_stride=row,
                      dtype=case["dtype"])
    state = {"module": module, "opts": opts, "tensors": (q, k, v, o), "o": o,
             "buffers": [tuple(_Buffer(t[i]) for t in (q, k, v, o)) for i in range(calls)], "stack": None}
    if case["graph"]:
        torch.cuda.synchronize()  # the graph's stream does not wait for the fills above

        def body():
            for bufs in state["buffers"]:
                nc.flash_launch(module, *bufs, opts, stream.handle)

        state["stack"] = _Stack(stream, body)
    return state


def run(state):
    if state["stack"] is not None:
        state["stack"]()
    else:
        for bufs in state["buffers"]:
            nc.flash_launch(state["module"], *bufs, state["opts"])
    return state["o"]


def work(case):
    calls, s, d = case["layers"], case["seq_len"], case["head_dim"]
    pairs = s * (s + 1) // 2 if case["causal"] else s * s
    return {"bytes": calls * case["batch_heads"] * s * d * (3 * 2 + 4),
            "flops": calls * case["batch_heads"] * pairs * d * 4}


def tolerance(case):
    # The probabilities are rounded to the element type (11 or 8 significant bits) before the PV
    # product, at a running maximum that implementations choose differently. Measured against exact()
    # over 26 cases: f16 rel 3e-5-2.1e-4, max 4.3e-3; bf16 rel 2.5e-4-1.4e-3, max 3.7e-2 (largest on
    # the early rows of causal cases, where few keys carry the weight). Four times the largest, and
    # somewhat more on rel, since two implementations are each off by that much.
    return {"rel": 7e-3, "max": 0.15} if case["dtype"] == "bf16" else {"rel": 1e-3, "max": 0.02}


def exact(case, seed):
    """The attention of the same inputs in float64, paddings of O as prepare() leaves them."""
    row, strides = _strides(case)
    bh, s, d, calls = case["batch_heads"], case["seq_len"], case["head_dim"], case["layers"]
    q, k, v = (t.as_strided((calls, bh, s, d), (bh * st, st, row, 1))
               for t, st in zip(_inputs(case, seed), strides))
    out = torch.zeros(calls, bh * strides[3], device="cuda", dtype=torch.float64)
    o = out.as_strided((calls, bh, s, d), (bh * strides[3], strides[3], row, 1))
    scale = 1.0 / math.sqrt(d)
    for c in range(calls):
        for b in range(bh):
            kt = k[c, b].double().t().contiguous()
            vb = v[c, b].double()
            for r0 in range(0, s, 4096):
                r1 = min(s, r0 + 4096)
                scores = (q[c, b, r0:r1].double() @ kt) * scale
                if case["causal"]:
                    keys = torch.arange(s, device="cuda")
                    rows = torch.arange(r0, r1, device="cuda")
                    scores.masked_fill_(keys[None, :] > rows[:, None], float("-inf"))
                o[c, b, r0:r1] = torch.softmax(scores, dim=1) @ vb
    return out
