"""What a user of this package has it do, as cases to be timed.

Six ways of calling the binary low-rank linear layer, each over the range of sizes it is used at:

``linear``         one `NanoQuantLinear.forward`, prepared for decode ("gemv") or prefill ("gemm"), called eagerly: the
                   drop-in use in existing model code.
``decode_layers``  a token step over decoder layers in the shape a decoder issues it, `decode_group` on {q,k,v}, {o},
                   {gate,up}, {down} of every layer, captured in a HIP graph once and replayed per token (a decode loop
                   under torch.compile(mode="reduce-overhead") is the same thing).
``decode_mixture`` the same for weights that are sums of two terms: `MixtureOfRankLinear.forward` per projection.
``decode_stack``   `DecodeRunList`: the linears of a whole stack in one launch.
``prefill_layer``  a prompt through the projections of one decoder layer: `prefill_group` on the same four groups.
``prefill_mixture`` the same for two-term weights.

Shapes are those of the package's own benchmarks (`nanoquant_amd.bench_decode.MODEL_SHAPES`), its 2048 x 2048 single
layer, and generic ones of the same ranges; ranks follow from the bits per weight.  Signs are i.i.d. (what a trained
factor looks like to the kernels), scales |N(0, 0.02)| + 1e-3, and activations N(0, 1) times a log-normal gain per
channel, since the channels of a hidden state differ in size.
"""
from __future__ import annotations

import math

import torch

from nanoquant_amd import DecodeRunList, MixtureOfRankLinear, NanoQuantLinear, decode_group, prefill_group
from nanoquant_amd.bench_decode import MODEL_SHAPES
from nanoquant_amd.packing import repack_words, tile_words

DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}
GROUPS = (("q", "k", "v"), ("o",), ("gate", "up"), ("down",))    # what a decoder layer issues, in this order


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: one module, one token; launches and host time are all there is
        dict(name="linear_decode_1_row", path="linear", kernel="gemv", m=2048, n=2048, bpw=1.0, rows=1, dtype="float16"),
        # one module on a ragged small batch (continuous batching), odd rank, bf16 as most checkpoints are
        dict(name="linear_decode_11_rows", path="linear", kernel="gemv", m=4096, n=11008, bpw=1.0, rows=11, dtype="bfloat16"),
        # single-stream generation: a token through eight decoder layers
        dict(name="layers_decode_1_row", path="decode_layers", model="llama2-7b", layers=8, bpw=1.0, rows=1, dtype="float16"),
        # a few sequences at once, grouped-query shapes, bf16, below one bit per weight
        dict(name="layers_decode_4_rows", path="decode_layers", model="qwen3-8b", layers=8, bpw=0.8, rows=4, dtype="bfloat16"),
        # two-term weights at 0.55 bits, one token
        dict(name="mixture_decode_1_row", path="decode_mixture", model="qwen3-8b", layers=4, bpw=0.55, rows=1, dtype="float16"),
        # the whole weight stream of a 7B stack in one launch
        dict(name="stack_decode_1_row", path="decode_stack", model="llama2-7b", layers=32, bpw=1.0, rows=1, dtype="float16"),
        # the same at the largest batch of the decode path
        dict(name="stack_decode_16_rows", path="decode_stack", model="llama2-7b", layers=32, bpw=1.0, rows=16, dtype="bfloat16"),
        # the largest: 8.6 GB of packed words, eight sequences
        dict(name="stack_decode_8_rows_70b", path="decode_stack", model="llama3-70b", layers=80, bpw=1.0, rows=8, dtype="float16"),
        # one module on a ragged prompt
        dict(name="linear_prefill_333_tokens", path="linear", kernel="gemm", m=11008, n=4096, bpw=1.0, rows=333, dtype="float16"),
        # a short prompt through a layer
        dict(name="layer_prefill_128_tokens", path="prefill_layer", model="llama2-7b", bpw=1.0, rows=128, dtype="float16"),
        # a long prompt, bf16
        dict(name="layer_prefill_4096_tokens", path="prefill_layer", model="llama2-7b", bpw=1.0, rows=4096, dtype="bfloat16"),
        # two-term weights on a prompt of ordinary length
        dict(name="mixture_prefill_512_tokens", path="prefill_mixture", model="qwen3-8b", bpw=0.55, rows=512, dtype="float16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["linear", "linear", "decode_layers", "decode_mixture", "decode_stack", "decode_stack",
                       "prefill_layer", "prefill_mixture"])
    dtype = rng.choice(["float16", "bfloat16"])
    bpw = round(rng.uniform(0.55, 1.0), 2)
    small = rng.choice(["llama2-7b", "qwen3-8b"])
    if path == "linear":
        # decode takes any width; the prefill layout wants n in 256s and m in 32s
        if rng.random() < 0.5:
            m, n = _log_int(rng, 1024, 28672), _log_int(rng, 1024, 28672)
            if rng.random() < 0.75:                       # hidden sizes are usually multiples of 64
                m, n = m // 64 * 64, n // 64 * 64
            return dict(path=path, kernel="gemv", m=m, n=n, bpw=bpw, rows=_log_int(rng, 1, 16), dtype=dtype)
        m, n = _log_int(rng, 1024, 13824) // 32 * 32, _log_int(rng, 1024, 13824) // 256 * 256
        return dict(path=path, kernel="gemm", m=m, n=n, bpw=bpw, rows=_log_int(rng, 128, 4096), dtype=dtype)
    if path == "decode_layers":
        return dict(path=path, model=small, layers=rng.randint(4, 9), bpw=bpw, rows=_log_int(rng, 1, 16), dtype=dtype)
    if path == "decode_mixture":
        return dict(path=path, model=small, layers=rng.randint(3, 8), bpw=bpw, rows=rng.choice([1, 1, 2, 4]), dtype=dtype)
    if path == "decode_stack":
        model = rng.choice(["llama2-7b", "qwen3-8b", "llama3-70b"])
        layers = _log_int(rng, 1, {"llama2-7b": 32, "qwen3-8b": 36, "llama3-70b": 40}[model])
        return dict(path=path, model=model, layers=layers, bpw=bpw, rows=rng.choice([1, 1, 2, 4, 8, 16]), dtype=dtype)
    model = small if path == "prefill_layer" else "qwen3-8b"
    return dict(path=path, model=model, bpw=min(bpw, 0.9), rows=_log_int(rng, 128, 4096), dtype=dtype)


# ---------------------------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------------------------
def _rank(m, n, bpw):
    """Rank at which r (m + n) sign bits are bpw bits per weight."""
    return max(32, int(round(bpw * m * n / (m + n))))


def _term_ranks(m, n, bpw):
    """Two terms, 3:1, each a whole number of packed words."""
    total = _rank(m, n, bpw)
    return [max(32, total * 3 // 4 // 32 * 32), max(32, total // 4 // 32 * 32)]


def _shapes(case):
    """[(m, n, [ranks])] of one layer (or of the one linear)."""
    if case["path"] == "linear":
        return [(case["m"], case["n"], [_rank(case["m"], case["n"], case["bpw"])])]
    two = case["path"].endswith("mixture")
    return [(m, n, _term_ranks(m, n, case["bpw"]) if two else [_rank(m, n, case["bpw"])]) for _, m, n in MODEL_SHAPES[case["model"]]]


def work(case):
    """Packed bits and scales once, every input once, every output once; two products per sign, row and term."""
    rows, nbytes, flops = case["rows"], 0.0, 0.0
    for m, n, ranks in _shapes(case):
        nbytes += 2.0 * rows * m
        for r in ranks:
            nbytes += r * (m + n) / 8 + 2 * (n + r + m)
            flops += 2.0 * rows * r * (m + n)
    # projections of one group read the same activations
    widths = [case["n"]] if case["path"] == "linear" else [_width(case["model"], g[0]) for g in GROUPS]
    nbytes += sum(2.0 * rows * n for n in widths)
    layers = case.get("layers", 1)
    return {"bytes": nbytes * layers, "flops": flops * layers}


def _width(model, name):
    return next(n for nm, _, n in MODEL_SHAPES[model] if nm == name)


def tolerance(case):
    # Against the same layer in 64 bits from the same packed words the paths differ by 2.2e-4 to 3.9e-4 (fp16) and
    # 1.7e-3 to 3.0e-3 (bf16): the roundings of the result, of h and of x * s_in to the 16-bit type.  Four times that.
    return {"rel": 1.5e-3} if case["dtype"] == "float16" else {"rel": 1.2e-2}


# ---------------------------------------------------------------------------------------------
# inputs, weights and plans
# ---------------------------------------------------------------------------------------------
class _Maker:
    def __init__(self, seed, dtype):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(seed)
        self.dtype = dtype

    def words(self, rows, cols):
        """Packed random signs [rows, ceil(cols / 32)] in the checkpoint's bit order, padding bits 0 (+1)."""
        w = torch.randint(-2 ** 31, 2 ** 31 - 1, (rows, (cols + 31) // 32), dtype=torch.int32, device=self.dev, generator=self.gen)
        if cols % 32:
            w[:, -1] &= (1 << (cols % 32)) - 1
        return w

    def scale(self, k):
        return (torch.randn(k, device=self.dev, generator=self.gen).abs() * 0.02 + 1e-3).to(self.dtype)

    def x(self, rows, n):
        gain = torch.exp(0.5 * torch.randn(n, device=self.dev, generator=self.gen))
        return (torch.randn(rows, n, device=self.dev, generator=self.gen) * gain).to(self.dtype)

    def module(self, m, n, r, kernel):
        """A module loaded from a packed checkpoint entry."""
        mod = NanoQuantLinear(n, m, r, device=self.dev, dtype=self.dtype)
        state = {"V_packed": self.words(r, n), "V_shape": torch.tensor([r, n]), "U_packed": self.words(m, r),
                 "U_shape": torch.tensor([m, r]), "scale_pre": self.scale(n)[None], "scale_mid": self.scale(r)[None],
                 "scale_post": self.scale(m)[None]}
        mod.load_packed(state, kernel_type=kernel, dtype=self.dtype)
        return mod

    def mixture(self, m, n, ranks, kernel):
        mix = MixtureOfRankLinear([self.module(m, n, r, kernel) for r in ranks])
        mix.kernel_type, mix.dtype = kernel, self.dtype
        return mix

    def layers(self, case, kernel):
        """Per layer a dict of its projections by name, and the input of every group."""
        make = self.mixture if case["path"].endswith("mixture") else lambda m, n, ranks, k: self.module(m, n, ranks[0], k)
        got = []
        for _ in range(case.get("layers", 1)):
            mods = {name: make(m, n, ranks, kernel)
                    for (name, _, _), (m, n, ranks) in zip(MODEL_SHAPES[case["model"]], _shapes(case))}
            got.append([([mods[name] for name in group], self.x(case["rows"], mods[group[0]].in_features)) for group in GROUPS])
        return got


def _captured(step):
    """`step` in a HIP graph, as a decode loop keeps it: (graph, its outputs)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    return graph, outs


def prepare(case, seed):
    mk = _Maker(seed, DTYPES[case["dtype"]])
    path, rows = case["path"], case["rows"]
    if path == "linear":
        mod = mk.module(case["m"], case["n"], _shapes(case)[0][2][0], case["kernel"])
        x = mk.x(rows, case["n"])
        return {"path": path, "mod": mod, "x": x if case["kernel"] == "gemv" else x[None]}
    if path in ("prefill_layer", "prefill_mixture"):
        return {"path": path, "groups": mk.layers(case, "gemm")[0]}
    if path in ("decode_layers", "decode_mixture"):
        layers = mk.layers(case, "gemv")
        if path == "decode_layers":
            step = lambda: [y for layer in layers for mods, x in layer for y in decode_group(mods, x)]
        else:
            step = lambda: [mod(x) for layer in layers for mods, x in layer for mod in mods]
        graph, outs = _captured(step)
        return {"path": path, "layers": layers, "graph": graph, "outs": outs}
    # decode_stack: every linear reads its group's input and writes its own piece of one output buffer
    shapes = _shapes(case)
    layers = case["layers"]
    out = torch.empty(rows * layers * sum(m for m, _, _ in shapes), dtype=mk.dtype, device=mk.dev)
    rl = DecodeRunList(rows, mk.dtype, mk.dev)
    at = 0
    for _ in range(layers):
        xs = {name: x for group in GROUPS for x in [mk.x(rows, _width(case["model"], group[0]))] for name in group}
        for (name, _, _), (m, n, (r,)) in zip(MODEL_SHAPES[case["model"]], shapes):
            rp = (r + 31) // 32 * 32                      # whole words; the padding has a zero mid scale
            s_mid = mk.scale(rp)
            s_mid[r:] = 0
            v, u = (tile_words(repack_words(w, "lsb_first", "half2")) for w in (mk.words(rp, n), mk.words(m, rp)))
            rl.add(xs[name], mk.scale(n), v, s_mid, u, mk.scale(m), y=out[at:at + rows * m].view(rows, m), tiled=True)
            at += rows * m
    rl.build()
    return {"path": path, "runlist": rl, "out": out}


def run(state):
    path = state["path"]
    if path == "linear":
        return state["mod"](state["x"])
    if path in ("prefill_layer", "prefill_mixture"):
        return [y for mods, x in state["groups"] for y in prefill_group(mods, x)]
    if path in ("decode_layers", "decode_mixture"):
        state["graph"].replay()
        return state["outs"]
    state["runlist"].run()
    return state["out"]
