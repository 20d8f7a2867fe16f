"""The work that a user has the framework do, as cases that can be timed and checked.

A case is one call (or one training step's calls) through the public Python entry
points of triton_metal.ops: `matmul`, `SAEEncoder` and `AttentionLayer`, with
operands resident in HBM.  `listed()` names the cases that stand for the whole
range, `draw()` gives more of the same ranges, `prepare()` makes a case's operands,
`run()` is one pass, `exact()` the same in 64 bits by plain torch.
"""

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "triton-metal_amd"))

from triton_metal import _core, ops  # noqa: E402
from triton_metal.buffer import DeviceBuffer  # noqa: E402

DTYPE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
NAME = {"f32": "float32", "f16": "float16", "bf16": "bfloat16"}


def listed():
    return [
        # The smallest call: one fp32 256^3 product (the first benchmark
        # configuration), a few microseconds of work behind one launch.
        {"name": "gemm_f32_256", "op": "gemm", "element": "f32", "layout": "nn",
         "m": 256, "n": 256, "k": 256, "pad": 0},
        # fp32 at sizes that are no multiple of anything: the ragged product of the
        # tests (129 x 257 x 65) sixteen, twelve and sixteen times over.
        {"name": "gemm_f32_odd", "op": "gemm", "element": "f32", "layout": "nn",
         "m": 2049, "n": 3079, "k": 1025, "pad": 0},
        # An ordinary 16-bit layer of a small model: 1024 tokens through a 1024 x 1024
        # projection stored as its weight (x @ W^T).
        {"name": "gemm_f16_1024", "op": "gemm", "element": "f16", "layout": "nt",
         "m": 1024, "n": 1024, "k": 1024, "pad": 0},
        # Decoding: 16 rows against an 8192 x 8192 weight, bound by reading the weight.
        {"name": "gemm_bf16_skinny", "op": "gemm", "element": "bf16", "layout": "nn",
         "m": 16, "n": 8192, "k": 8192, "pad": 0},
        # The large square product (the benchmark's GEMM configuration).
        {"name": "gemm_bf16_8192", "op": "gemm", "element": "bf16", "layout": "nn",
         "m": 8192, "n": 8192, "k": 8192, "pad": 0},
        # 16-bit at odd sizes, so rows of A, B and C start at any 2-byte address: a
        # vocabulary or feature count that nobody padded.
        {"name": "gemm_bf16_odd", "op": "gemm", "element": "bf16", "layout": "nn",
         "m": 2049, "n": 4097, "k": 1025, "pad": 0},
        # The sparse-autoencoder encoder at the benchmark's size.
        {"name": "sae_bf16", "op": "sae", "element": "bf16", "m": 8192, "k": 2048, "n": 16384},
        # The host training loop's step (2 heads of 96 rows, fp32): forward and
        # backward of a tiny layer, bound by launches and latency.
        {"name": "attn_f32_small", "op": "attn", "element": "f32", "train": True,
         "causal": False, "heads": 2, "seq": 96, "dim": 64},
        # fp32 training at the largest published fp32 attention size.
        {"name": "attn_f32_2048", "op": "attn", "element": "f32", "train": True,
         "causal": False, "heads": 16, "seq": 2048, "dim": 64},
        # bf16 causal training at the headline configuration (B4 H32 S4096 D128).
        {"name": "attn_bf16_4096", "op": "attn", "element": "bf16", "train": True,
         "causal": True, "heads": 128, "seq": 4096, "dim": 128},
        # The other usual head size, f16, B8 H16 S1024 D64 (the benchmark's forward
        # configuration) as a training step.
        {"name": "attn_f16_d64", "op": "attn", "element": "f16", "train": True,
         "causal": False, "heads": 128, "seq": 1024, "dim": 64},
        # A head size between the usual two (80, as in the tests) and a sequence that
        # is no multiple of a tile, causal, bf16.
        {"name": "attn_bf16_d80", "op": "attn", "element": "bf16", "train": True,
         "causal": True, "heads": 32, "seq": 1000, "dim": 80},
    ]


#: Most operations of a drawn case: the listed products' 1.1e12 for 16-bit elements
#: in whole rows, less where the arithmetic is fp32 or the sizes are odd, so that none
#: takes longer than the largest listed one.
_MOST_FLOPS = 1.0e12
_MOST_FLOPS_SLOW = {"attn": 2.5e10, "gemm": 5.0e10, "sae": 5.0e10}


def _size(rng, low, high, odd):
    """A size spread over its logarithm; multiples of 64 or 8, or any number."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    step = 1 if odd else rng.choice((8, 64))
    return max(1 if odd else step, int(round(v / step)) * step)


def draw(rng):
    op = rng.choice(("gemm", "gemm", "gemm", "sae", "attn", "attn", "attn"))
    element = rng.choice(("bf16", "bf16", "f16", "f32"))
    if op == "attn":
        dim = rng.choice((32, 64, 64, 80, 96, 128, 128))
        slow = element == "f32" or dim not in (64, 128)
        while True:
            case = {"op": op, "element": element, "train": rng.random() < 0.7,
                    "causal": rng.random() < 0.6,
                    "heads": int(round(math.exp(rng.uniform(0.0, math.log(128))))),
                    "seq": _size(rng, 64, 4096, rng.random() < 0.4), "dim": dim}
            if work(case)["flops"] <= (_MOST_FLOPS_SLOW[op] if slow else _MOST_FLOPS):
                return case
    odd = rng.random() < 0.4
    while True:
        m, n, k = _size(rng, 16, 8192, odd), _size(rng, 64, 16384, odd), _size(rng, 64, 8192, odd)
        case = {"op": op, "element": element, "m": m, "n": n, "k": k}
        if op == "gemm":
            case["layout"] = rng.choice(("nn", "nn", "nt", "tn"))
            case["pad"] = rng.choice((0, 0, 8, 1))  # elements between one stored row and the next
        slow = element == "f32" or odd or case.get("pad", 0) % 8
        if work(case)["flops"] <= (_MOST_FLOPS_SLOW[op] if slow else _MOST_FLOPS):
            return case


# --------------------------------------------------------------------------- #
# Library buffers as torch tensors
# --------------------------------------------------------------------------- #

_ADDRESS = r"""
extern "C" __global__ void address_of(void *buffer, unsigned long long *out) {
  if (threadIdx.x == 0) *out = (unsigned long long)buffer;
}
"""
_address = {}


def _device_address(buffer):
    """A buffer's address in HBM, told by a user kernel that is given the buffer."""
    if not _address:
        _address["library"] = _core.compile_msl(_ADDRESS)
        _address["kernel"] = _core.load_kernel(_address["library"], "address_of")
        _address["out"] = DeviceBuffer((1,), "uint64")
    out = _address["out"]
    _core.launch(_address["kernel"], (1, 1, 1), 64, [_core.ARG_BUFFER] * 2,
                 [buffer.tm_handle, out.tm_handle])
    return int(out.numpy()[0])


class _Owner:
    """Frees what it holds once neither the state nor a tensor over it is left."""

    def __init__(self, *things):
        self.things = things

    def __del__(self):
        try:
            _core.synchronize()
            for t in self.things:
                t.free()
        except Exception:  # the interpreter is ending
            pass


class _Memory:
    _TYPES = {2: "<i2", 4: "<f4"}

    def __init__(self, buffer, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {
            "shape": (buffer.numel,), "typestr": self._TYPES[buffer.itemsize],
            "data": (_device_address(buffer), False), "version": 2}


def _tensor(buffer, owner):
    """The buffer's memory as a torch tensor of its shape and type, without a copy."""
    flat = torch.as_tensor(_Memory(buffer, owner), device="cuda")
    return flat.view(getattr(torch, buffer.dtype)).view(buffer.shape)


# --------------------------------------------------------------------------- #
# Inputs
# --------------------------------------------------------------------------- #


def _normal(shape, element, generator, scale=1.0):
    x = torch.randn(shape, generator=generator, device="cuda", dtype=torch.float32)
    return x.mul_(scale).to(DTYPE[element])


def _inputs(case, seed):
    """Operands by name, in the order drawn: activations and upstream gradients
    N(0, 1), weights N(0, 1/K) as initialised or trained layers have them."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)
    e = case["element"]
    if case["op"] == "attn":
        shape = (case["heads"], case["seq"], case["dim"])
        return {name: _normal(shape, e, g) for name in ("q", "k", "v", "do")}
    m, n, k = case["m"], case["n"], case["k"]
    got = {"a": _normal((m, k), e, g), "b": _normal((k, n), e, g, 1.0 / math.sqrt(k))}
    if case["op"] == "sae":
        got["bias"] = _normal((n,), e, g, 0.1)
    return got


def _stored(x, pad):
    """[rows, cols + pad] with x in the first columns and zeros behind."""
    return torch.nn.functional.pad(x, (0, pad)) if pad else x.contiguous()


def prepare(case, seed):
    """What a program holds before the call: operands in library buffers, an output
    buffer, the layer or encoder object."""
    x = _inputs(case, seed)
    e = case["element"]
    if case["op"] == "attn":
        layer = ops.AttentionLayer(case["heads"], case["seq"], case["dim"], e, case["causal"])
        owner = _Owner(layer)
        for name, value in x.items():
            _tensor(layer.buffers[name], owner).copy_(value)
        names = ("o", "lse") + (("dq", "dk", "dv") if case["train"] else ())
        torch.cuda.synchronize()
        return {"layer": layer, "owner": owner, "train": case["train"], "op": "attn",
                "out": {name: _tensor(layer.buffers[name], owner) for name in names}}
    m, n, k = case["m"], case["n"], case["k"]
    if case["op"] == "sae":
        shapes = {"a": (m, k), "b": (k, n), "bias": (n,)}
        stored = x
        out_shape = (m, n)
    else:
        pad, layout = case["pad"], case["layout"]
        a = x["a"].t() if layout == "tn" else x["a"]
        b = x["b"].t() if layout == "nt" else x["b"]
        stored = {"a": _stored(a, pad), "b": _stored(b, pad)}
        shapes = {name: tuple(t.shape) for name, t in stored.items()}
        out_shape = (m, n + pad)
        lda, ldb = shapes["a"][1], shapes["b"][1]
        strides = ((1, lda) if layout == "tn" else (lda, 1)) + \
            ((1, ldb) if layout == "nt" else (ldb, 1)) + (n + pad, 1)
    buffers = {name: DeviceBuffer(shape, NAME[e]) for name, shape in shapes.items()}
    c = DeviceBuffer(out_shape, NAME[e])
    owner = _Owner(*buffers.values(), c)
    for name, value in stored.items():
        _tensor(buffers[name], owner).copy_(value)
    out = _tensor(c, owner)
    out.zero_()
    torch.cuda.synchronize()
    state = {"op": case["op"], "buffers": buffers, "c": c, "owner": owner, "out": out[:, :n]}
    if case["op"] == "sae":
        state["encoder"] = ops.SAEEncoder(e)
    else:
        state["size"], state["strides"] = (m, n, k), strides
    return state


def run(state):
    """One pass, queued as a program queues it that does not wait for each call."""
    if state["op"] == "gemm":
        b = state["buffers"]
        ops.matmul(b["a"], b["b"], state["c"], *state["size"], strides=state["strides"],
                   synchronous=False)
    elif state["op"] == "sae":
        b = state["buffers"]
        state["encoder"](b["a"], b["b"], b["bias"], state["c"], synchronous=False)
    else:
        state["layer"].run_forward(synchronous=False)
        if state["train"]:
            state["layer"].run_backward(synchronous=False)
    return state["out"]


def work(case):
    size = 4 if case["element"] == "f32" else 2
    if case["op"] == "attn":
        h, s, d = case["heads"], case["seq"], case["dim"]
        pairs = h * s * (s + 1) / 2 if case["causal"] else h * s * s
        # Q, K, V in and O, L out; with a backward dO in, dQ, dK, dV out
        tensors = 8 if case["train"] else 4
        return {"bytes": tensors * h * s * d * size + h * s * 4,
                "flops": (14 if case["train"] else 4) * pairs * d}
    m, n, k = case["m"], case["n"], case["k"]
    bias = n if case["op"] == "sae" else 0
    return {"bytes": (m * k + k * n + m * n + bias) * size, "flops": 2 * m * n * k}


def tolerance(case):
    """About four times the distance from 64 bits: a product's is its result's
    rounding, attention's also that of P and dS, which the kernels hold in the
    element type where they feed a product."""
    if case["op"] == "attn":
        return {"rel": {"f32": 1e-5, "f16": 1.2e-3, "bf16": 1e-2}[case["element"]]}
    return {"rel": {"f32": 1e-5, "f16": 1e-3, "bf16": 8e-3}[case["element"]]}


def exact(case, seed):
    """The outputs of `run` in 64 bits, from the same rounded operands."""
    x = {name: value.double() for name, value in _inputs(case, seed).items()}
    if case["op"] != "attn":
        c = x["a"] @ x["b"]
        return torch.relu(c + x["bias"]) if case["op"] == "sae" else c
    scale = 1.0 / math.sqrt(case["dim"])
    seq = case["seq"]
    names = ("o", "lse") + (("dq", "dk", "dv") if case["train"] else ())
    got = {name: [] for name in names}
    hidden = torch.ones((seq, seq), dtype=torch.bool, device="cuda").triu(1)
    for h in range(case["heads"]):
        q, k, v, do = (x[name][h] for name in ("q", "k", "v", "do"))
        s = (q @ k.t().contiguous()) * scale
        if case["causal"]:
            s.masked_fill_(hidden, -math.inf)
        lse = torch.logsumexp(s, -1)
        p = torch.exp(s - lse[:, None])
        o = p @ v
        got["o"].append(o)
        got["lse"].append(lse / math.log(2.0))  # the kernels keep it in log2 units
        if case["train"]:
            delta = (do * o).sum(-1)
            ds = p * (do @ v.t().contiguous() - delta[:, None])
            got["dq"].append(ds @ k * scale)
            got["dk"].append(ds.t().contiguous() @ q * scale)
            got["dv"].append(p.t().contiguous() @ do)
    return {name: torch.stack(v) for name, v in got.items()}
