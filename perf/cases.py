"""The performance cases of the quantized-linear inference path.

Every case is work that a model lowered with ``AutoKernelLowering`` does in a forward step, eagerly, through the
lowered modules.  Four kinds:

``linear``  one quantized linear layer on ``tokens`` rows of activations.  ``scheme`` is ``vq`` (codebook of ``nc`` rows
            of eight fp16 values), ``rvq`` (main codebook of ``nc`` rows, residual codebook of 256, an fp16 scale
            and offset per output row) or ``q`` (``nbits``-bit codes with an fp16 scale per ``group``, with or without zero points).
``block``   the lowered modules of one decoder block: two RMSNorms and the q / k / v / o / gate / up / down linears.
            Attention and the gated activation are the model's own code, so what they would hand to ``o`` and ``down`` is an input.
``tables``  the lookups in front of the first block: a VQ embedding, an int4 embedding and one RMSNorm.

Shapes come from the benchmark configurations; ``draw`` ranges over what lies between them: 1 to 4096 tokens (decode
steps of a batch at the low end, prompts at the high end), 256 to 14336 features, fp16 and bf16, codebooks of
16 to 65536 rows, uniform and Zipf(1.1) indices, biases, column permutations, ragged sizes.
"""

import math

import torch

DEVICE = "cuda"
VL = 8  # values per codebook vector
MAX_WORK = 2.0 * 4096 * 14336 * 4096  # operations of the largest case


def _linear(name, scheme, n, k, tokens, dtype, **more):
    case = {"name": name, "kind": "linear", "scheme": scheme, "n": n, "k": k, "tokens": tokens, "dtype": dtype, "bias": False}
    case.update({"nc": 65536, "zipf": False, "perm": False} if scheme == "vq" else
                {"nc": 65536, "zipf": True} if scheme == "rvq" else
                {"nbits": 4, "group": 32, "zero_point": False})  # fmt: skip
    case.update(more)
    return case


def _block(name, hidden, inter, kv, tokens, dtype, nc):
    return {"name": name, "kind": "block", "hidden": hidden, "inter": inter, "kv": kv, "tokens": tokens, "dtype": dtype, "nc": nc}


def listed():
    return [
        # The smallest call there is: an up-projection of a 270M model, one decode token.
        _linear("vq8-small-m1", "vq", 2048, 640, 1, "float16", nc=256),
        # A decode step of a 1B model's block, 12-bit indices: nine short launches one behind the other.
        _block("vq12-block-m1", 2048, 8192, 512, 1, "float16", 4096),
        # A decode step of an 8B model's block, 16-bit indices: the decode path that serving spends its time in.
        _block("vq16-block-m1", 4096, 14336, 1024, 1, "bfloat16", 65536),
        # Sixteen sequences decoded together, the long reduction of a down-projection.
        _linear("vq16-down-m16", "vq", 4096, 14336, 16, "bfloat16"),
        # A short prompt, or one slice of a chunked one, through an up-projection.
        _linear("vq16-up-m384", "vq", 14336, 4096, 384, "bfloat16"),
        # A long prompt through the same layer: the largest call.
        _linear("vq16-up-m4096", "vq", 14336, 4096, 4096, "bfloat16"),
        # Residual VQ, attention projection, decode and prompt.
        _linear("rvq-m1", "rvq", 4096, 4096, 1, "float16"),
        _linear("rvq-m384", "rvq", 4096, 4096, 384, "float16"),
        # Group-quantized int4, decode and prompt.
        _linear("q4-m1", "q", 14336, 4096, 1, "float16"),
        _linear("q4-m256", "q", 14336, 4096, 256, "float16"),
        # Nothing a multiple of a tile: odd rows, 10-bit indices, columns permuted, a bias, K not a multiple of 64.
        _linear("vq10-ragged-m77", "vq", 3003, 2184, 77, "float16", nc=1000, bias=True, perm=True),
        # Embedding lookups and the first norm of a long prompt.
        {"name": "tables-m4096", "kind": "tables", "vocab": 128256, "dim": 4096, "tokens": 4096, "dtype": "bfloat16", "nc": 65536},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, step):
    return max(step, int(round(_log(rng, lo, hi) / step)) * step)


def draw(rng):
    dtype = rng.choice(["float16", "bfloat16"])
    tokens = int(round(_log(rng, 1, 4096)))
    kind = rng.choices(["vq", "q", "rvq", "block", "tables"], [45, 25, 12, 10, 8])[0]
    if kind == "block":
        hidden = _size(rng, 512, 4096, 128)
        inter, kv = _size(rng, 2 * hidden, min(14336, 4 * hidden), 128), hidden // rng.choice([1, 2, 4])
        case = _block("", hidden, inter, kv, tokens, dtype, rng.choice([256, 4096, 65536]))
        case["tokens"] = max(1, min(tokens, int(MAX_WORK / work(case)["flops"] * tokens)))
    elif kind == "tables":
        case = {"kind": "tables", "vocab": _size(rng, 4096, 128256, 1), "dim": _size(rng, 256, 4096, 64), "tokens": tokens,
                "dtype": dtype, "nc": rng.choice([256, 4096, 65536])}  # fmt: skip
    else:
        n = _size(rng, 256, 14336, rng.choice([1, 16, 64, 128]))
        step = 128 if kind == "q" else rng.choice([8, 64, 128, 256])
        k = _size(rng, 256, 14336, step)
        tokens = max(1, min(tokens, int(MAX_WORK / (2.0 * n * k))))
        case = _linear("", kind, n, k, tokens, dtype, bias=rng.random() < 0.25)
        if kind == "vq":
            nc = rng.choice([256, 1024, 4096, 16384, 65536, int(_log(rng, 16, 65536))])
            case.update(nc=nc, zipf=rng.random() < 0.3, perm=rng.random() < 0.2)
        elif kind == "rvq":
            case.update(nc=rng.choice([4096, 65536]), zipf=rng.random() < 0.6)
        else:
            case.update(nbits=rng.choice([4, 4, 4, 8]), group=rng.choice([32, 64, 128]), zero_point=rng.random() < 0.3)
    case.pop("name", None)
    return case


# ----------------------------------------------------------------------------------------------------------------------
# What a program has in hand before the call: the lowered model on its GPU, and the activations.
# ----------------------------------------------------------------------------------------------------------------------


def _indices(g, nc, count, zipf):
    if not zipf:
        return torch.randint(0, nc, (count,), generator=g, device=DEVICE)
    p = torch.arange(1, nc + 1, dtype=torch.float64, device=DEVICE) ** -1.1
    edges = torch.cumsum(p / p.sum(), 0)
    u = torch.rand(count, generator=g, device=DEVICE, dtype=torch.float64)
    return torch.searchsorted(edges, u).clamp_(max=nc - 1)


def _codebook(g, rows):
    return (torch.randn(rows, VL, generator=g, device=DEVICE) * 0.02).to(torch.float16)


def _vq_weight(g, case, n, k, cb):
    from neuropress_amd.qweights import VQWeight

    count = n * (k // VL)
    bits = 0
    if cb.shape[0] <= 16 and count % 2:
        bits = 8  # a 4-bit stream holds an even number of indices
    idx = _indices(g, cb.shape[0], count, case.get("zipf", False))
    perm = torch.randperm(k, generator=g, device=DEVICE) if case.get("perm") else None
    return VQWeight.from_indices(idx, cb, n, k, column_permutation=perm, bits=bits)


def _rvq_weight(g, case, n, k):
    from neuropress_amd.qweights import VQScheme, VQWeight
    from neuropress_amd.transforms.vq_packing import IndexPacking

    count = n * (k // VL)
    cb, cr = _codebook(g, case["nc"]), _codebook(g, 256)
    main, res = (_indices(g, rows, count, case["zipf"]) for rows in (case["nc"], 256))
    scheme = VQScheme(
        centroids=cb, original_shape=(n, k), residual_centroids=cr,
        row_scale=(torch.rand(n, generator=g, device=DEVICE) + 0.5).to(torch.float16),
        row_bias=(torch.randn(n, generator=g, device=DEVICE) * 0.01).to(torch.float16),
    )  # fmt: skip
    return VQWeight(IndexPacking.pack(main, scheme.is_packed_indices), scheme, IndexPacking.pack(res, scheme.residual_bits))


def _q_weight(g, n, k, nbits, group, zero_point, dtype):
    from neuropress_amd.qweights import ScalarQScheme, ScalarQWeight

    blob = torch.randint(0, 256, (n, k * nbits // 8), generator=g, device=DEVICE, dtype=torch.uint8)
    scale = (torch.rand(n * (k // group), generator=g, device=DEVICE) * 0.019 + 0.001).to(torch.float16)
    zp = None
    if zero_point:
        zp = torch.randint(0, 1 << nbits, (n * (k // group),), generator=g, device=DEVICE).to(torch.float16)
    return ScalarQWeight(blob, ScalarQScheme(nbits, group, scale, zp), dtype)


def _module(weight, n, k, bias=None):
    from neuropress_amd.qweights import attach_quantized_weight

    linear = torch.nn.Linear(k, n, bias=False, device="meta")
    attach_quantized_weight(linear, weight)
    if bias is not None:
        linear.bias = torch.nn.Parameter(bias, requires_grad=False)
    return linear


def _norm(g, dim, dtype):
    norm = torch.nn.RMSNorm(dim, eps=1e-5, device=DEVICE, dtype=dtype)
    norm.weight.requires_grad_(False)
    norm.weight.copy_(1 + 0.1 * torch.randn(dim, generator=g, device=DEVICE))
    return norm


def _lower(model):
    from neuropress_amd import AutoKernelLowering

    AutoKernelLowering().apply(model)
    return model


class _Block(torch.nn.Module):
    def forward(self, x, attention, residual, activated):
        h = self.norm1(x)
        q, k, v = self.q(h), self.k(h), self.v(h)
        o = self.o(attention)
        h = self.norm2(residual)
        gate, up = self.gate(h), self.up(h)
        return q, k, v, o, gate, up, self.down(activated)


class _Tables(torch.nn.Module):
    def forward(self, ids):
        a, b = self.vq(ids), self.q4(ids)
        return a, b, self.norm(a)


def _block_shapes(case):
    h, f, kv = case["hidden"], case["inter"], case["kv"]
    return {"q": (h, h), "k": (kv, h), "v": (kv, h), "o": (h, h), "gate": (f, h), "up": (f, h), "down": (h, f)}


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = getattr(torch, case["dtype"])
    tokens = case["tokens"]

    def activations(dim):  # decode: one token of each sequence of the batch; longer: one prompt
        shape = (tokens, 1, dim) if tokens <= 16 else (1, tokens, dim)
        return torch.randn(shape, generator=g, device=DEVICE).to(dtype)

    if case["kind"] == "block":
        model, cb = _Block(), _codebook(g, case["nc"])
        for name, (n, k) in _block_shapes(case).items():
            setattr(model, name, _module(_vq_weight(g, case, n, k, cb), n, k))
        model.norm1, model.norm2 = (_norm(g, case["hidden"], dtype) for _ in range(2))
        h, f = case["hidden"], case["inter"]
        return _lower(model), (activations(h), activations(h), activations(h), activations(f))

    if case["kind"] == "tables":
        from neuropress_amd.qweights import attach_quantized_weight

        model, vocab, dim = _Tables(), case["vocab"], case["dim"]
        for name, weight in (("vq", _vq_weight(g, case, vocab, dim, _codebook(g, case["nc"]))),
                             ("q4", _q_weight(g, vocab, dim, 4, 32, False, dtype))):  # fmt: skip
            table = torch.nn.Embedding(vocab, dim, device="meta")
            setattr(model, name, attach_quantized_weight(table, weight))
        model.norm = _norm(g, dim, dtype)
        ids = torch.randint(0, vocab, (1, tokens), generator=g, device=DEVICE)
        return _lower(model), (ids,)

    n, k = case["n"], case["k"]
    if case["scheme"] == "vq":
        weight = _vq_weight(g, case, n, k, _codebook(g, case["nc"]))
    elif case["scheme"] == "rvq":
        weight = _rvq_weight(g, case, n, k)
    else:
        weight = _q_weight(g, n, k, case["nbits"], case["group"], case["zero_point"], dtype)
    bias = torch.randn(n, generator=g, device=DEVICE).to(dtype) if case["bias"] else None
    model = _lower(torch.nn.Sequential(_module(weight, n, k, bias)))
    return model[0], (activations(k),)


def run(state):
    model, inputs = state
    return model(*inputs)


# ----------------------------------------------------------------------------------------------------------------------
# What a pass cannot do without, and how near two implementations come.
# ----------------------------------------------------------------------------------------------------------------------


def _bits(rows):
    return max(4, (rows - 1).bit_length())


def work(case):
    tokens = case["tokens"]
    if case["kind"] == "tables":
        dim, nc = case["dim"], case["nc"]
        rows = min(tokens, case["vocab"])
        read = rows * (dim // VL * 2 + dim // 2 + dim // 32 * 2) + min(nc, rows * dim // VL) * VL * 2 + tokens * 8 + dim * 2
        return {"bytes": read + 3 * tokens * dim * 2, "flops": 8.0 * tokens * dim}
    if case["kind"] == "block":
        shapes = _block_shapes(case)
        pairs = sum(n * k for n, k in shapes.values())
        nbytes = pairs // VL * _bits(case["nc"]) / 8 + case["nc"] * VL * 2
        nbytes += 2 * tokens * (sum(n for n, _ in shapes.values()) + 3 * case["hidden"] + case["inter"]) + 4 * case["hidden"]
        return {"bytes": nbytes, "flops": 2.0 * tokens * pairs}
    n, k = case["n"], case["k"]
    if case["scheme"] == "q":
        nbytes = n * k * case["nbits"] / 8 + n * (k // case["group"]) * (4 if case["zero_point"] else 2)
    else:
        nbytes = n * k // VL * _bits(case["nc"]) / 8 + case["nc"] * VL * 2
        if case["scheme"] == "rvq":
            nbytes += n * k // VL + 256 * VL * 2 + 4 * n
        if case.get("perm"):
            nbytes += 4 * k
    nbytes += 2 * tokens * (n + k) + (2 * n if case["bias"] else 0)
    return {"bytes": nbytes, "flops": 2.0 * tokens * n * k}


def tolerance(case):
    # Outputs are rounded to 11 (fp16) or 8 (bf16) significant bits, and so is the decoded weight; sums are f32.
    if case["dtype"] == "bfloat16":
        return {"rel": 5e-3, "max": 3e-2}
    return {"rel": 1e-3, "max": 5e-3}
