"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values with a "kind":

  linear    one ``QuantizedLinear`` called eagerly, as a module of any model: the smallest calls
  stack     the quantized linears of a few decoder layers for one decode step, grouped as a decoder calls them
            (q/k/v, o, gate/up, down) and replayed from one HIP graph, as a serving loop does
  step      a whole greedy-decode step of ``StaticDecoder`` (embedding to logits, KV cache included), graph-replayed
  prefill   the quantized linears of a decoder layer over a prompt's rows, called eagerly
  quantize  ``quantize_linear`` of one layer with its calibration Hessian
  encode    ``codebook.quantize`` over many 8-vectors (scale fitting, rounding a whole weight to nearest)
  export    a quantized layer back to its dense weight: ``dequantize_linear`` and ``reconstruct_weight``

Every layer of a stack reads an input of its own, so that a rounding difference in one layer does not travel through
the others.  Codes follow the codeword frequencies of Gaussian weights, activations have the heavy channels of real
hidden states.
"""
import itertools
import math
import types

import torch

from quipsharp_amd.checkpoint import QuantizedLinear, grouped_forward
from quipsharp_amd.codebooks import E8OneBitCodebook, E8PCodebook
from quipsharp_amd.decode import StaticDecoder
from quipsharp_amd.incoherence import IncoherenceSigns, KronSigns
from quipsharp_amd.quantize import QuantizedLayer, RVQCodebookAdapter, dequantize_linear, quantize_linear
from quipsharp_amd.rvq import RVQStage

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# hidden size, intermediate size, query width, key / value width, attention bias: decoder layers that the benchmark names
LAYERS = {
    "llama2_7b": (4096, 11008, 4096, 4096, False),
    "llama3_8b": (4096, 14336, 4096, 1024, False),
    "qwen25_7b": (3584, 18944, 3584, 512, True),
    "qwen3_32b": (5120, 25600, 8192, 1024, False),
}
STAGE_SCALES = {"2bit": (1.0,), "3bit": (0.95, 0.55), "4bit": (0.95, 0.28)}
INPUT_SCALE = {"2bit": 0.96, "3bit": 1.0, "4bit": 1.0}  # what a weight of unit variance is divided by


def listed():
    return [
        # the smallest call: one row through a key projection, the module called eagerly
        dict(name="linear_1row", kind="linear", m=1024, n=4096, bits="2bit", rows=1, dtype="bf16", bias=False,
             transform="rht"),
        # a layer of a checkpoint written with the FFT transform (odd sizes), a few rows
        dict(name="linear_rfft_4rows", kind="linear", m=11008, n=4096, bits="2bit", rows=4, dtype="bf16", bias=False,
             transform="rfft"),
        # batch-1 decode of the largest model that the benchmark has
        dict(name="decode_1row", kind="stack", model="qwen3_32b", bits="2bit", layers=4, rows=1, dtype="bf16"),
        # decode of a few sequences, two residual stages
        dict(name="decode_5rows_3bit", kind="stack", model="llama3_8b", bits="3bit", layers=4, rows=5, dtype="bf16"),
        # a whole step of a small batch over a long context
        dict(name="step_4x4000", kind="step", layers=2, rows=4, pos=3999, max_len=4352),
        # a short ragged prompt, two residual stages, fp16
        dict(name="prefill_45_3bit", kind="prefill", model="llama3_8b", bits="3bit", layers=2, rows=45, dtype="fp16"),
        # an ordinary prompt
        dict(name="prefill_512", kind="prefill", model="llama2_7b", bits="2bit", layers=2, rows=512, dtype="bf16"),
        # the longest prompt, widths with odd factors and an attention bias
        dict(name="prefill_4000", kind="prefill", model="qwen25_7b", bits="2bit", layers=1, rows=4000, dtype="bf16"),
        # quantizing: the square layer of a 7B model
        dict(name="quantize_4096", kind="quantize", m=4096, n=4096, bits="2bit", tune=10),
        # quantizing: a narrow layer with odd factors, two stages
        dict(name="quantize_ragged_3bit", kind="quantize", m=1024, n=3584, bits="3bit", tune=4),
        # rounding many vectors to the nearest codeword
        dict(name="encode_1m", kind="encode", vectors=1 << 20, bits="2bit"),
        # a dense weight from its codes
        dict(name="export_4096x11008", kind="export", m=4096, n=11008, bits="2bit"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "stack", "stack", "step", "prefill", "prefill", "quantize", "encode",
                       "export"])
    bits = rng.choice(["2bit", "2bit", "3bit"])
    if kind == "linear":
        transform = rng.choice(["rht", "rht", "rht", "rfft"])
        # also sizes off the 16 x 256 tiles, and odd factors from 3 to 43
        sizes = [256, 384, 640, 896, 1024, 1536, 2560, 3584, 4096, 5120, 8192, 11008, 14336, 18944, 25600]
        return dict(kind=kind, m=rng.choice(sizes), n=rng.choice(sizes), bits=bits, rows=_log_int(rng, 1, 33),
                    dtype=rng.choice(["bf16", "fp16", "fp32"]), bias=rng.random() < 0.3, transform=transform)
    if kind == "stack":
        return dict(kind=kind, model=rng.choice(sorted(LAYERS)), bits=bits, layers=rng.choice([2, 3, 4]),
                    rows=_log_int(rng, 1, 16), dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "step":
        pos = _log_int(rng, 64, 6000)
        return dict(kind=kind, layers=rng.choice([1, 2]), rows=rng.randint(1, 8), pos=pos,
                    max_len=pos + rng.randint(1, 300))
    if kind == "prefill":
        return dict(kind=kind, model=rng.choice(sorted(LAYERS)), bits=bits, layers=1, rows=_log_int(rng, 17, 2500),
                    dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "quantize":
        return dict(kind=kind, m=rng.choice([1024, 1536, 2048, 3584, 4096]),
                    n=rng.choice([1024, 1536, 2048, 2560, 3584] if bits == "2bit" else [1024, 1536, 2048, 2560]),
                    bits=bits, tune=rng.choice([0, 1, 4, 8] if bits == "2bit" else [0, 1, 2, 4]))
    if kind == "encode":
        return dict(kind=kind, vectors=_log_int(rng, 2000, 1 << 20), bits=rng.choice(["1bit", "2bit", "3bit", "4bit"]))
    return dict(kind=kind, m=rng.choice([512, 1024, 3584, 4096, 5120, 8192]),
                n=rng.choice([1024, 2560, 4096, 11008, 14336]), bits=rng.choice(["2bit", "3bit", "4bit"]))


# ----------------------------------------------------------------------------
# the codebooks' tables in plain Python, for the frequencies of codes and for the 64-bit results
# ----------------------------------------------------------------------------
_PAD = """31113333 13113333 11313333 11133333 33313311 33313131 33311331 33313113 33311313 33311133 33133311 33133131
33131331 33133113 33131313 33131133 31333311 31333131 31331331 31333113 31331313 13331133 13333311 13333131 13331331
13333113 13331313 11331333 33113331""".split()
_TABLES = {}


def _tables():
    """(E8P table of absolute values with the sign of the last coordinate, E8 one-bit table), fp64 on the GPU."""
    if not _TABLES:
        rows = []

        def grow(row, budget):
            if len(row) == 8:
                rows.append(row)
                return
            for k in range(4):
                if k * (k + 1) <= budget:
                    grow(row + [k + 0.5], budget - k * (k + 1))

        grow([], 8)
        rows += [[int(d) / 2 for d in word] for word in _PAD]
        rows = [r[:7] + [-r[7] if int(sum(r)) % 2 else r[7]] for r in rows]
        one = [[0.0] * 8]
        one += [list(v) for v in itertools.product((-1.0, 0.0, 1.0), repeat=8)
                if sum(x * x for x in v) == 2]
        one += [list(v) for v in itertools.product((-0.5, 0.5), repeat=8) if sum(v) % 2 == 0]
        four = (v for v in itertools.product((-2.0, -1.0, 0.0, 1.0, 2.0), repeat=8)
                if sum(x * x for x in v) == 4 and sum(v) % 2 == 0)
        one += [list(v) for v in itertools.islice(four, 15)]
        assert len(rows) == 256 and len(one) == 256
        _TABLES["e8p"] = torch.tensor(rows, dtype=torch.float64, device=DEV)
        _TABLES["one"] = torch.tensor(one, dtype=torch.float64, device=DEV)
    return _TABLES["e8p"], _TABLES["one"]


def _decode64(codes, bits):
    """fp64 values (..., 8) of codes (stages, ...) of a residual chain."""
    e8p, one = _tables()
    total = 0.0
    for s, scale in enumerate(STAGE_SCALES[bits]):
        c = codes[s].to(torch.int64) & 0xFFFF
        if s == 1 and bits == "3bit":
            v = one[c & 0xFF]
        else:
            flips = (c.unsqueeze(-1) >> torch.arange(7, 0, -1, device=DEV)) & 1
            flips = torch.cat([flips, flips.sum(-1, keepdim=True) & 1], -1)
            v = e8p[c >> 8] * (1 - 2 * flips) + ((c & 1).double() * 0.5 - 0.25).unsqueeze(-1)
        total = total + v * scale
    return total


def _codes(gen, shape, bits):
    """int16 codes (stages, *shape) with the frequencies that a Gaussian weight's codes have."""
    e8p, one = _tables()
    count = math.prod(shape)
    out = []
    for s in range(len(STAGE_SCALES[bits])):
        table = one if s == 1 and bits == "3bit" else e8p
        weight = torch.exp(-0.4 * table.square().sum(1)).float().cpu()
        edges = (weight / weight.sum()).cumsum(0).to(DEV)
        row = torch.searchsorted(edges, torch.rand(count, generator=gen, device=DEV)).clamp_(max=255)
        if table is e8p:
            row = (row << 8) | torch.randint(0, 256, (count,), generator=gen, device=DEV)
        out.append(((row + 32768) % 65536 - 32768).to(torch.int16).view(*shape))
    return torch.stack(out)


def _codebook(bits):
    if bits == "1bit":
        return E8OneBitCodebook(DEV)
    first = E8PCodebook(DEV)
    if bits == "2bit":
        return first
    second = E8OneBitCodebook(DEV) if bits == "3bit" else E8PCodebook(DEV)
    s0, s1 = STAGE_SCALES[bits]
    return RVQCodebookAdapter([RVQStage(first, s0), RVQStage(second, s1)])


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _signs(gen, n):
    return torch.randint(0, 2, (n,), generator=gen, device=DEV).float() * 2 - 1


def _activations(gen, rows, n, dtype):
    """Hidden states: unit variance, a few channels far above the rest."""
    heavy = torch.rand(n, generator=gen, device=DEV)
    scale = torch.where(heavy < 0.004, 12.0, 0.6 + 0.8 * torch.rand(n, generator=gen, device=DEV))
    return (torch.randn(rows, n, generator=gen, device=DEV) * scale).to(DTYPES[dtype])


def _pow2(n):
    return n & (n - 1) == 0


def _module(gen, m, n, bits, bias=False, transform="rht"):
    """A QuantizedLinear as a loaded checkpoint has it."""
    kind = transform if transform == "rfft" else "rht" if _pow2(m) and _pow2(n) else "krht"
    q = QuantizedLinear(n, m, 8, kind, num_stages=len(STAGE_SCALES[bits]), has_bias=bias).to(DEV)
    codes = _codes(gen, (m, n // 8), bits)
    q.codes.copy_(codes[0] if codes.shape[0] == 1 else codes)
    q.scale.fill_(0.0135 * math.sqrt(4096 / n))
    if kind == "rfft":
        for name, size in (("phase_u", m // 2), ("phase_v", n // 2)):
            angle = 2 * math.pi * torch.rand(size, generator=gen, device=DEV)
            getattr(q, name).copy_(torch.polar(torch.ones_like(angle), angle))
    else:
        q.su.copy_(_signs(gen, m))
        q.sv.copy_(_signs(gen, n))
    if bias:
        q.bias.copy_(torch.randn(m, generator=gen, device=DEV) * 0.1)
    q.codebook = _codebook(bits)
    return q


def _groups(model):
    """[(input width, [(output width, bias)])] of a decoder layer's calls."""
    hidden, inter, qw, kvw, bias = LAYERS[model]
    return [(hidden, [(qw, bias), (kvw, bias), (kvw, bias)]), (qw, [(hidden, False)]),
            (hidden, [(inter, False), (inter, False)]), (inter, [(hidden, False)])]


def _layer_inputs(case, gen):
    """[(x, [modules])] for every call of every layer."""
    calls = []
    for _ in range(case["layers"]):
        for n, outs in _groups(case["model"]):
            mods = [_module(gen, m, n, case["bits"], bias) for m, bias in outs]
            calls.append((_activations(gen, case["rows"], n, case["dtype"]), mods))
    return calls


def _call(calls):
    out = []
    for x, mods in calls:
        out += grouped_forward(x, mods) if len(mods) > 1 else [mods[0](x)]
    return out


def _capture(fn):
    """fn captured in a HIP graph after a warm-up outside it: (graph, fn's outputs)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


# ----------------------------------------------------------------------------
# a decoder with the shapes of the benchmark's largest model, for whole steps
# ----------------------------------------------------------------------------
VOCAB, HEADS, KV_HEADS, HEAD_DIM, EPS, THETA = 32768, 64, 8, 128, 1e-6, 1e6


class _Weight(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = weight


class _Embedding(_Weight):
    def forward(self, ids):
        return torch.nn.functional.embedding(ids, self.weight)


class _Head(_Weight):
    def forward(self, x):
        return torch.nn.functional.linear(x, self.weight)


def _rotary(x, pos):
    freq = THETA ** (-torch.arange(0, HEAD_DIM, 2, device=DEV).float() / HEAD_DIM)
    angle = pos[..., None].float() * freq
    angle = torch.cat([angle, angle], -1)
    return angle.cos().to(x.dtype), angle.sin().to(x.dtype)


def _norm_weight(gen, n):
    return _Weight((1 + 0.1 * torch.randn(n, generator=gen, device=DEV)).bfloat16())


def _decoder(case, gen):
    hidden, inter, qw, kvw, _ = LAYERS["qwen3_32b"]
    make = lambda m, n: _module(gen, m, n, "2bit")  # noqa: E731
    layers = []
    for _ in range(case["layers"]):
        attn = types.SimpleNamespace(q_proj=make(qw, hidden), k_proj=make(kvw, hidden), v_proj=make(kvw, hidden),
                                     o_proj=make(hidden, qw), q_norm=_norm_weight(gen, HEAD_DIM),
                                     k_norm=_norm_weight(gen, HEAD_DIM))
        mlp = types.SimpleNamespace(gate_proj=make(inter, hidden), up_proj=make(inter, hidden),
                                    down_proj=make(hidden, inter))
        layers.append(types.SimpleNamespace(self_attn=attn, mlp=mlp, input_layernorm=_norm_weight(gen, hidden),
                                            post_attention_layernorm=_norm_weight(gen, hidden)))
    rand = lambda *s: (0.02 * torch.randn(*s, generator=gen, device=DEV)).bfloat16()  # noqa: E731
    inner = types.SimpleNamespace(layers=layers, embed_tokens=_Embedding(50 * rand(VOCAB, hidden)),
                                  norm=_norm_weight(gen, hidden), rotary_emb=_rotary)
    config = types.SimpleNamespace(num_attention_heads=HEADS, num_key_value_heads=KV_HEADS, head_dim=HEAD_DIM,
                                   hidden_size=hidden, rms_norm_eps=EPS)
    model = types.SimpleNamespace(model=inner, config=config, lm_head=_Head(rand(VOCAB, hidden)))
    dec = StaticDecoder(model, case["rows"], case["max_len"])
    for cache in dec.k + dec.v:  # the context so far
        cache[:, :, :case["pos"]] = torch.randn(case["rows"], KV_HEADS, case["pos"], HEAD_DIM, generator=gen,
                                                device=DEV).bfloat16()
    ids = torch.randint(0, VOCAB, (case["rows"], 1), generator=gen, device=DEV)
    return dec, ids, torch.full((1,), case["pos"], dtype=torch.int64, device=DEV)


# ----------------------------------------------------------------------------
# prepare / run
# ----------------------------------------------------------------------------
def _quantize_inputs(case, gen):
    m, n = case["m"], case["n"]
    W = 0.02 * torch.randn(m, n, generator=gen, device=DEV) * (
        0.7 + 0.6 * torch.rand(m, 1, generator=gen, device=DEV))
    # calibration rows with heavy channels and correlated columns
    mix = torch.randn(n, 64, generator=gen, device=DEV) / 8
    X = _activations(gen, 4096, n, "fp32") + torch.randn(4096, 64, generator=gen, device=DEV) @ mix.T
    return W, X.T @ X / 4096


def _encode_input(case, gen):
    x = torch.randn(case["vectors"], 8, generator=gen, device=DEV)
    return x / INPUT_SCALE.get(case["bits"], 1.0)


def _export_layer(case, gen):
    m, n = case["m"], case["n"]
    codes = _codes(gen, (m, n // 8), case["bits"]).to(torch.int64) & 0xFFFF
    cls = IncoherenceSigns if _pow2(m) and _pow2(n) else KronSigns
    signs = cls(su=_signs(gen, m), sv=_signs(gen, n))
    return QuantizedLayer(codes=codes[0] if codes.shape[0] == 1 else codes, signs=signs, g=8, shape=(m, n),
                          scale=0.0135)


def prepare(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind == "linear":
        q = _module(gen, case["m"], case["n"], case["bits"], case["bias"], case["transform"])
        x = _activations(gen, case["rows"], case["n"], case["dtype"])
        return {"run": lambda: q(x)}
    if kind == "stack":
        calls = _layer_inputs(case, gen)
        graph, out = _capture(lambda: _call(calls))
        return {"run": lambda: (graph.replay(), out)[1], "keep": calls}
    if kind == "step":
        dec, ids, pos = _decoder(case, gen)
        graph, logits = _capture(lambda: dec.step(ids, pos))
        return {"run": lambda: (graph.replay(), [logits] + dec.k + dec.v)[1], "keep": (dec, ids, pos)}
    if kind == "prefill":
        calls = _layer_inputs(case, gen)
        return {"run": lambda: _call(calls)}
    codebook = _codebook(case["bits"])
    if kind == "quantize":
        W, H = _quantize_inputs(case, gen)

        def quantize():
            layer, what = quantize_linear(W, H, codebook, generator=torch.Generator().manual_seed(int(seed)),
                                          codebook_scale=INPUT_SCALE[case["bits"]], tune_iters=case["tune"])
            return {"codes": layer.codes, "su": layer.signs.su, "sv": layer.signs.sv, "scale": layer.scale,
                    "what": what}
        return {"run": quantize}
    if kind == "encode":
        x = _encode_input(case, gen)
        return {"run": lambda: codebook.quantize(x)}
    layer = _export_layer(case, gen)
    return {"run": lambda: layer.signs.reconstruct_weight(dequantize_linear(layer, codebook))}


def run(state):
    with torch.no_grad():
        return state["run"]()


# ----------------------------------------------------------------------------
# work and tolerances
# ----------------------------------------------------------------------------
def _linear_work(m, n, rows, bits, elem):
    """Codes once (2 bytes per 8 weights, 1 more for the one-bit stage), the rows in and out."""
    per8 = {"2bit": 2, "3bit": 3, "4bit": 4}[bits]
    return m * n // 8 * per8 + elem * rows * (m + n) + (m + n) // 8, 2 * rows * m * n


def work(case):
    kind = case["kind"]
    b = f = 0
    if kind == "linear":
        b, f = _linear_work(case["m"], case["n"], case["rows"], case["bits"], 4 if case["dtype"] == "fp32" else 2)
    elif kind in ("stack", "prefill", "step"):
        model, bits = case.get("model", "qwen3_32b"), case.get("bits", "2bit")
        for n, outs in _groups(model):
            for m, _ in outs:
                one = _linear_work(m, n, case["rows"], bits, 2)
                b, f = b + one[0], f + one[1]
        b, f = b * case["layers"], f * case["layers"]
        if kind == "step":
            hidden = LAYERS[model][0]
            keys = case["layers"] * case["rows"] * (case["pos"] + 1) * HEAD_DIM
            b += 2 * 2 * KV_HEADS * keys + 2 * VOCAB * (hidden + case["rows"])
            f += 4 * HEADS * keys + 2 * case["rows"] * VOCAB * hidden
    elif kind == "quantize":
        # W and H in, codes and the dense result out; the feedback products of the passes (each column of the error
        # with the rest), the factorization and the transforms' butterflies
        m, n, t = case["m"], case["n"], case["tune"]
        b = 4 * (2 * m * n + n * n) + 8 * len(STAGE_SCALES[case["bits"]]) * m * n // 8
        f = m * n * n + 2 * t * m * n * n + n ** 3 // 3 + (m * n + n * n) * int(math.log2(max(m, n))) * 2
    elif kind == "encode":
        stages = 1 if case["bits"] in ("1bit", "2bit") else 2
        b = case["vectors"] * (32 + 32 + 8 * stages)
        f = case["vectors"] * stages * 2 * 8 * 256
    else:
        m, n = case["m"], case["n"]
        b = 8 * len(STAGE_SCALES[case["bits"]]) * m * n // 8 + 4 * m * n
        f = m * n * int(math.log2(m * n))
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind == "encode":
        return "exact"  # the codes and values of the nearest codewords, bit for bit
    if kind == "export":
        # Walsh-Hadamard stages in one order, bit for bit; an odd factor is a short fp32 sum
        return "exact" if _pow2(case["m"]) and _pow2(case["n"]) else {"rel": 2e-6, "max": 1e-5}
    if kind == "quantize":
        # a rounding difference of 1e-7 in the feedback moves a near-tie now and then, and the rest of that row with
        # it: with the refinement's sums in another order, up to 8e-5 of the codes and 4.5e-3 of the result at two
        # bits, and 2.2e-3 / 1.4e-2 at three (its second stage has many codewords of nearly equal distance)
        if case["bits"] == "2bit":
            return {"rel": 0.02, "max": 0.99, "differ": 0.002}
        return {"rel": 0.03, "max": 0.99, "differ": 0.01}
    if kind == "step":
        return {"rel": 2e-2, "max": 0.3}
    if case.get("dtype") == "fp32":
        return {"rel": 1e-3, "max": 1e-2}  # fp16 operands
    return {"rel": 6e-3, "max": 5e-2} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 2e-2}


# ----------------------------------------------------------------------------
# the same results in 64 bits
# ----------------------------------------------------------------------------
def _transform64(x):
    """The orthonormal transform of the last axis, K_p (x) H_L with K_p the discrete Hartley matrix, in fp64."""
    n = x.shape[-1]
    L = n & -n
    p = n // L
    y = x.double().reshape(-1, p, L)
    h = 1
    while h < L:
        v = y.view(-1, p, L // (2 * h), 2, h)
        y = torch.stack([v[..., 0, :] + v[..., 1, :], v[..., 0, :] - v[..., 1, :]], -2).view(-1, p, L)
        h *= 2
    y = y / math.sqrt(L)
    if p > 1:
        a = torch.arange(p, dtype=torch.float64, device=x.device)
        angle = 2 * math.pi / p * torch.remainder(a[:, None] * a[None, :], p)
        K = (angle.cos() + angle.sin()) / math.sqrt(p)
        y = (y.transpose(1, 2).reshape(-1, p) @ K).view(-1, L, p).transpose(1, 2)
    return y.reshape(x.shape)


def _fft64(x, phase, inverse):
    z = torch.view_as_complex(x.double().reshape(*x.shape[:-1], -1, 2).contiguous())
    phase = phase.to(torch.complex128)
    z = torch.fft.ifft(z, norm="ortho") * phase.conj() if inverse else torch.fft.fft(z * phase, norm="ortho")
    return torch.view_as_real(z).reshape(x.shape)


def _linear64(q, x):
    codes = q.codes if q.codes.dim() == 3 else q.codes.unsqueeze(0)
    bits = "2bit" if codes.shape[0] == 1 else "3bit"
    W = _decode64(codes, bits).reshape(q.out_features, q.in_features) * q.scale.double()
    if q.transform_kind == "rfft":
        y = _fft64(_fft64(x, q.phase_v, False) @ W.T, q.phase_u, True)
    else:
        y = _transform64(_transform64(x.double() * q.sv.double()) @ W.T) * q.su.double()
    return y if q.bias is None else y + q.bias.double()


def _rms64(h, weight):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def _step64(case, seed):
    dec, ids, pos = _decoder(case, _gen(seed))
    model, B, p = dec.model.model, case["rows"], case["pos"]
    cos, sin = (t[p].double() for t in (dec.cos, dec.sin))
    h = model.embed_tokens(ids)[:, 0].double()
    ks, vs = [], []
    for i, L in enumerate(model.layers):
        a = L.self_attn
        x = _rms64(h, L.input_layernorm.weight)
        q = _rope64(_rms64(_linear64(a.q_proj, x).view(B, HEADS, HEAD_DIM), a.q_norm.weight), cos, sin)
        k = _rope64(_rms64(_linear64(a.k_proj, x).view(B, KV_HEADS, HEAD_DIM), a.k_norm.weight), cos, sin)
        K, V = dec.k[i].double(), dec.v[i].double()
        K[:, :, p], V[:, :, p] = k, _linear64(a.v_proj, x).view(B, KV_HEADS, HEAD_DIM)
        score = (K[:, :, None, :p + 1] * q.view(B, KV_HEADS, -1, 1, HEAD_DIM)).sum(-1) * dec.scale
        o = (torch.softmax(score, -1)[..., None] * V[:, :, None, :p + 1]).sum(-2).reshape(B, -1)
        h = h + _linear64(a.o_proj, o)
        x = _rms64(h, L.post_attention_layernorm.weight)
        h = h + _linear64(L.mlp.down_proj, torch.nn.functional.silu(_linear64(L.mlp.gate_proj, x)) *
                          _linear64(L.mlp.up_proj, x))
        ks.append(K)
        vs.append(V)
    return [_rms64(h, model.norm.weight) @ dec.model.lm_head.weight.double().T] + ks + vs


def _nearest64(x, kind):
    """Nearest codewords of fp64 x (N, 8): the least distance over tables, shifts and even numbers of sign flips."""
    e8p, one = _tables()
    if kind == "one":
        return one[torch.cat([(c[:, None] - one).square().sum(-1).argmin(1) for c in x.split(1 << 15)])]
    out = []
    for c in x.split(1 << 14):
        best = None
        for shift in (-0.25, 0.25):
            xs = (c - shift)[:, None]
            prod = xs * e8p
            gap = prod.abs().min(-1)
            odd = (prod < 0).sum(-1) & 1
            d = (xs.square() + e8p.square() - 2 * prod.abs()).sum(-1) + 4 * odd * gap.values
            d, row = d.min(1)
            at = row[:, None]
            sign = torch.where(prod.gather(1, at[..., None].expand(-1, 1, 8))[:, 0] < 0, -1.0, 1.0)
            flip = torch.nn.functional.one_hot(gap.indices.gather(1, at)[:, 0], 8) * odd.gather(1, at)
            v = e8p[row] * sign * (1 - 2 * flip) + shift
            best = (d, v) if best is None else (torch.minimum(best[0], d),
                                                torch.where((d < best[0])[:, None], v, best[1]))
        out.append(best[1])
    return torch.cat(out)


def exact(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind == "linear":
        q = _module(gen, case["m"], case["n"], case["bits"], case["bias"], case["transform"])
        return _linear64(q, _activations(gen, case["rows"], case["n"], case["dtype"]))
    if kind in ("stack", "prefill"):
        return [_linear64(q, x) for x, mods in _layer_inputs(case, gen) for q in mods]
    if kind == "step":
        return _step64(case, seed)
    if kind == "quantize":
        # the codes depend on every rounding before them; the scale is the weight's own
        W, _ = _quantize_inputs(case, gen)
        return {"codes": None, "su": None, "sv": None, "what": None,
                "scale": float(W.double().square().mean().sqrt() * INPUT_SCALE[case["bits"]])}
    if kind == "encode":
        x = _encode_input(case, gen).double()
        if case["bits"] == "1bit":
            return [_nearest64(x, "one"), None]
        total = torch.zeros_like(x)
        for s, scale in enumerate(STAGE_SCALES[case["bits"]]):
            total += scale * _nearest64((x - total) / scale, "one" if s == 1 and case["bits"] == "3bit" else "e8p")
        return [total, None]
    layer = _export_layer(case, gen)
    m, n = layer.shape
    codes = layer.codes if layer.codes.dim() == 3 else layer.codes.unsqueeze(0)
    W = _decode64(codes, case["bits"]).reshape(m, n) * layer.scale
    W = _transform64(_transform64(W.T.contiguous()).T.contiguous())
    return W * layer.signs.su.double()[:, None] * layer.signs.sv.double()[None, :]
