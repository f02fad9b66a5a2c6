"""The performance cases of this package: what a structure-prediction model calls, through the public operators.

A case is a dict of plain values; ``kind`` names the operator it times:

* ``triangle``: ``triangle_attention`` on an N x N pair representation, starting or ending node;
* ``msa``: ``pair_bias_attention`` over the rows of an MSA, the pair bias shared by the rows;
* ``single``: ``gated_pair_bias_attention`` on the single representation (one row: latency counts);
* ``gate``: ``gate_attention_output``, the gated output stage behind MSA attention;
* ``trimul``: ``triangle_multiplication`` with mask and biases;
* ``norm``: ``layer_norm`` over pair rows.

``train`` runs the forward and the backward of every operand, else the forward of an inference call.  Crops of
training are multiples of 64; whole chains have any length.  Activations are unit normal (what follows a
LayerNorm and a projection), projection weights normal over the square root of their fan-in.
"""

from __future__ import annotations

import torch

import oops_amd

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # a small complex in float32, inference: the smallest call, launches and host time count
        dict(name="tri_64_f32", kind="triangle", n=64, h=4, d=32, ending=False, mask=False, dtype="f32", train=False),
        # a training crop with padded residues, starting node
        dict(name="tri_384_pad", kind="triangle", n=384, h=4, d=32, ending=False, mask=True, dtype="bf16", train=True),
        # the large training crop, ending node read in place: the headline workload
        dict(name="tri_768_end", kind="triangle", n=768, h=4, d=32, ending=True, mask=False, dtype="bf16", train=True),
        # a whole chain of odd length with unresolved residues masked, fine-tuned
        dict(name="tri_331_odd", kind="triangle", n=331, h=4, d=32, ending=False, mask=True, dtype="bf16", train=True),
        # float32 training on a small chain, ending node
        dict(name="tri_193_f32", kind="triangle", n=193, h=4, d=32, ending=True, mask=False, dtype="f32", train=True),
        # MSA row attention of a training crop: 512 sequences, 15% of the entries masked
        dict(name="msa_512x384", kind="msa", s=512, n=384, h=8, d=32, mask=True, dtype="bf16", train=True),
        # MSA row attention of a whole chain, float16 inference
        dict(name="msa_127x277_f16", kind="msa", s=127, n=277, h=8, d=32, mask=True, dtype="f16", train=False),
        # gated attention of the single representation (16 heads of 24 channels), training
        dict(name="single_384", kind="single", n=384, h=16, d=24, mask=True, dtype="bf16", train=True),
        # the gated output stage behind MSA row attention, training
        dict(name="gate_512x384", kind="gate", s=512, n=384, h=8, d=32, dtype="bf16", train=True),
        # triangle multiplication of a training crop
        dict(name="trimul_512", kind="trimul", n=512, c=128, direction="outgoing", dtype="bf16", train=True),
        # triangle multiplication of a whole chain, inference
        dict(name="trimul_381_odd", kind="trimul", n=381, c=128, direction="incoming", dtype="bf16", train=False),
        # the pair LayerNorm of a 512-residue crop, training
        dict(name="norm_512", kind="norm", rows=512 * 512, width=128, dtype="bf16", train=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case: training crops half of the time a multiple of 64, everything else any length."""

    kind = rng.choice(["triangle", "triangle", "triangle", "msa", "msa", "single", "gate", "trimul", "trimul", "norm"])
    train = rng.random() < 0.6
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])

    def length(lo, hi):
        n = _log_int(rng, lo, hi)
        return max(64, n // 64 * 64) if train and rng.random() < 0.5 else n

    if kind == "triangle":
        n = length(48, 224 if dtype == "f32" else 640)
        return dict(kind=kind, n=n, h=4, d=32, ending=rng.random() < 0.5, mask=rng.random() < 0.5, dtype=dtype,
                    train=train)
    if kind == "msa":
        f32 = dtype == "f32"
        return dict(kind=kind, s=_log_int(rng, 16, 64 if f32 else 384), n=length(64, 192 if f32 else 384), h=8, d=32,
                    mask=rng.random() < 0.8, dtype=dtype, train=train)
    if kind == "single":
        return dict(kind=kind, n=length(64, 768), h=16, d=rng.choice([24, 24, 48, 64]), mask=rng.random() < 0.5,
                    dtype=rng.choice(["bf16", "bf16", "f32"]), train=train)
    if kind == "gate":
        return dict(kind=kind, s=_log_int(rng, 1, 512), n=length(64, 384), h=8, d=32, dtype=dtype, train=train)
    if kind == "trimul":
        return dict(kind=kind, n=length(48, 288 if dtype == "f32" else 512), c=rng.choice([64, 128, 128]),
                    direction=rng.choice(["incoming", "outgoing"]), dtype=dtype, train=train)
    n = _log_int(rng, 64, 512)
    return dict(kind=kind, rows=n * n, width=rng.choice([64, 128, 128, 256]), dtype=dtype, train=train)


# ----------------------------------------------------------------- inputs


class _Maker:
    """Normal tensors on the GPU from one seed."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def randn(self, *shape, scale=1.0):
        return (torch.randn(*shape, generator=self.g, device="cuda") * scale).to(self.dtype)

    def rand(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")


TRIMUL_WEIGHTS = (
    "input_norm_weight", "input_norm_bias", "left_value_weight", "left_gate_weight", "right_value_weight",
    "right_gate_weight", "output_norm_weight", "output_norm_bias", "output_weight", "output_gate_weight",
    "left_value_bias", "left_gate_bias", "right_value_bias", "right_gate_bias", "output_bias", "output_gate_bias",
)  # fmt: skip


def _inputs(case, seed):
    """The operands by name (every floating one but ``dout`` and ``pair_mask`` takes part in training)."""

    kind = case["kind"]
    m = _Maker(seed, DTYPES[case["dtype"]])
    if kind == "triangle":
        n, h, d = case["n"], case["h"], case["d"]
        names = ("query", "key", "value") + (("dout",) if case["train"] else ())
        x = {name: m.randn(1, n, n, h, d) for name in names}
        if case["ending"]:
            x = {name: t.transpose(1, 2) for name, t in x.items()}
        x["bias"] = m.randn(1, 1, h, n, n)
        if case["mask"]:
            # the last 10-30% of the residues are padding
            keep = n - round(n * (0.1 + 0.2 * float(m.rand(1))))
            row = torch.arange(n, device="cuda") < keep
            x["mask"] = (row[:, None] & row[None, :])[None]
        return x
    if kind in ("msa", "single"):
        s, n, h, d = case.get("s", 1), case["n"], case["h"], case["d"]
        # (rows, tokens, heads, head size) from a projection, viewed head-major
        x = {name: m.randn(s, n, h, d).transpose(1, 2) for name in ("query", "key", "value")}
        x["bias"] = m.randn(1, h, n, n)
        if case["mask"]:
            x["mask"] = m.rand(s, n) > 0.15
            x["mask"][:, 0] = True
        if kind == "msa":
            if case["train"]:
                x["dout"] = m.randn(s, h, n, d)
            return x
        c = h * d
        x["single"] = m.randn(s, n, c)
        x["gate_weight"] = m.randn(c, c, scale=c**-0.5)
        x["output_weight"] = m.randn(c, c, scale=c**-0.5)
        if case["train"]:
            x["dout"] = m.randn(s, n, c)
        return x
    if kind == "gate":
        s, n, h, d = case["s"], case["n"], case["h"], case["d"]
        c = h * d
        x = {"attention": m.randn(s, n, h, d).transpose(1, 2), "single": m.randn(s, n, c),
             "gate_weight": m.randn(c, c, scale=c**-0.5), "output_weight": m.randn(c, c, scale=c**-0.5)}
        if case["train"]:
            x["dout"] = m.randn(s, n, c)
        return x
    if kind == "trimul":
        n, c = case["n"], case["c"]
        x = {"pair": m.randn(1, n, n, c)}
        keep = torch.arange(n, device="cuda") < n - n // 8
        x["pair_mask"] = (keep[:, None] & keep[None, :])[None].float()
        for name in TRIMUL_WEIGHTS:
            if name.endswith("norm_weight"):
                x[name] = 1.0 + m.randn(c, scale=0.1)
            elif name.endswith("_bias"):
                x[name] = m.randn(c, scale=0.1)
            else:
                x[name] = m.randn(c, c, scale=c**-0.5)
        if case["train"]:
            x["dout"] = m.randn(1, n, n, c)
        return x
    rows, width = case["rows"], case["width"]
    x = {"input": m.randn(rows, width)}
    m.dtype = torch.float32  # the affine parameters stay float32
    x["weight"] = 1.0 + m.randn(width, scale=0.1)
    x["bias"] = m.randn(width, scale=0.1)
    if case["train"]:
        m.dtype = DTYPES[case["dtype"]]
        x["dout"] = m.randn(rows, width)
    return x


def _leaves(x):
    return [t for name, t in x.items() if name not in ("dout", "mask", "pair_mask")]


def prepare(case, seed):
    x = _inputs(case, seed)
    if case["train"]:
        for t in _leaves(x):
            t.requires_grad_(True)
    return case, x


# ----------------------------------------------------------------- the timed calls


def _call(case, x):
    kind = case["kind"]
    if kind == "triangle":
        return oops_amd.triangle_attention(x["query"], x["key"], x["value"], x.get("mask"), x["bias"])
    if kind == "msa":
        return oops_amd.pair_bias_attention(x["query"], x["key"], x["value"], x.get("mask"), x["bias"])
    if kind == "single":
        return oops_amd.gated_pair_bias_attention(x["single"], x["query"], x["key"], x["value"], x.get("mask"),
                                                  x["bias"], x["gate_weight"], x["output_weight"])
    if kind == "gate":
        return oops_amd.gate_attention_output(x["attention"], x["single"], x["gate_weight"], x["output_weight"])
    if kind == "trimul":
        weights = {name: x[name] for name in TRIMUL_WEIGHTS}
        return oops_amd.triangle_multiplication(x["pair"], x["pair_mask"], direction=case["direction"], **weights)
    return oops_amd.layer_norm(x["input"], case["width"], x["weight"], x["bias"])


def run(state):
    case, x = state
    if not case["train"]:
        with torch.no_grad():
            return _call(case, x)
    out = _call(case, x)
    return (out.detach(), *torch.autograd.grad(out, _leaves(x), x["dout"]))


# ----------------------------------------------------------------- what a pass cannot do without


def _attention_work(s, n, h, d, mask, el, train):
    rows = s * n * h * d * el
    bias = h * n * n * el
    keep = s * n if mask else 0
    lse = s * n * h * 4
    nbytes = 4 * rows + bias + keep  # q, k, v read, o written
    flops = 4 * s * h * d * n * n
    if train:
        # the log-sum-exp crosses from the forward to the backward, which reads q, k, v, o, do and
        # writes dq, dk, dv, dbias
        nbytes += 8 * rows + 2 * bias + keep + 2 * lse
        flops += 10 * s * h * d * n * n
    return nbytes, flops


def _gate_work(rows, c, el, train):
    nbytes = (3 * rows * c + 2 * c * c) * el  # attention, single, weights read, output written
    flops = 4 * rows * c * c
    if train:
        nbytes += (5 * rows * c + 4 * c * c) * el  # dout, attention, single read, two gradients written
        flops += 8 * rows * c * c
    return nbytes, flops


def work(case):
    kind, train = case["kind"], case["train"]
    el = 4 if case["dtype"] == "f32" else 2
    if kind == "triangle":
        n = case["n"]
        nbytes, flops = _attention_work(n, n, case["h"], case["d"], case["mask"], el, train)
    elif kind == "msa":
        nbytes, flops = _attention_work(case["s"], case["n"], case["h"], case["d"], case["mask"], el, train)
    elif kind == "single":
        c = case["h"] * case["d"]
        nbytes, flops = _attention_work(1, case["n"], case["h"], case["d"], case["mask"], el, train)
        gb, gf = _gate_work(case["n"], c, el, train)
        nbytes, flops = nbytes + gb, flops + gf
    elif kind == "gate":
        nbytes, flops = _gate_work(case["s"] * case["n"], case["h"] * case["d"], el, train)
    elif kind == "trimul":
        n, c = case["n"], case["c"]
        cells = n * n
        nbytes = (2 * cells * c + 6 * c * c) * el + 4 * cells
        flops = 2 * cells * c * 6 * c + 2 * c * n**3
        if train:
            nbytes += (3 * cells * c + 12 * c * c) * el + 4 * cells
            flops *= 3
    else:
        cells = case["rows"] * case["width"]
        nbytes = 2 * cells * el
        flops = 8 * cells
        if train:
            nbytes += 3 * cells * el
            flops += 16 * cells
    return {"bytes": nbytes, "flops": flops}


# ----------------------------------------------------------------- float64 reference


def _exact_attention(q, k, v, mask, bias, dout):
    """q, k, v (rows, H, N, D) float64; mask (rows, N); bias (H, N, N): (out, dq, dk, dv, dbias), rows in chunks."""

    rows, h, n, d = q.shape
    chunk = max(1, int(2.0e8 // (h * n * n)))
    parts, dbias = [], torch.zeros_like(bias)
    for r in range(0, rows, chunk):
        qc, kc, vc = q[r : r + chunk], k[r : r + chunk], v[r : r + chunk]
        logits = qc @ kc.transpose(-1, -2).contiguous()
        logits = logits.mul_(d**-0.5).add_(bias)
        if mask is not None:
            logits.masked_fill_(~mask[r : r + chunk, None, None, :], float("-inf"))
        p = torch.nan_to_num_(torch.softmax(logits, -1))  # a row without a kept key is zero
        del logits
        out = p @ vc
        if dout is None:
            parts.append((out,))
            continue
        doc = dout[r : r + chunk]
        dv = p.transpose(-1, -2).contiguous() @ doc
        ds = (doc @ vc.transpose(-1, -2).contiguous()).sub_((out * doc).sum(-1, keepdim=True)).mul_(p)
        dbias += ds.sum(0)
        parts.append((out, (ds @ kc) * d**-0.5, (ds.transpose(-1, -2).contiguous() @ qc) * d**-0.5, dv))
    cat = [torch.cat(t) for t in zip(*parts)]
    return cat if dout is None else [*cat, dbias]


def _exact_gate(att, single, wg, wo):
    return (torch.sigmoid(single @ wg.t()) * att.transpose(1, 2).flatten(2)) @ wo.t()


def _exact_trimul(x, direction):
    norm = torch.nn.functional.layer_norm
    pair, mask = x["pair"], x["pair_mask"][..., None]
    c = pair.shape[-1]
    lin = lambda t, name: t @ x[name + "_weight"].t() + x[name + "_bias"]  # noqa: E731
    xn = norm(pair, (c,), x["input_norm_weight"], x["input_norm_bias"])
    left = mask * lin(xn, "left_value") * torch.sigmoid(lin(xn, "left_gate"))
    right = mask * lin(xn, "right_value") * torch.sigmoid(lin(xn, "right_gate"))
    left, right = (t.permute(0, 3, 1, 2).contiguous() for t in (left, right))  # (1, C, N, N)
    if direction == "outgoing":
        comb = left @ right.transpose(-1, -2)
    else:
        comb = left.transpose(-1, -2) @ right
    nrm = norm(comb.permute(0, 2, 3, 1), (c,), x["output_norm_weight"], x["output_norm_bias"])
    return lin(nrm, "output") * torch.sigmoid(lin(xn, "output_gate"))


def exact(case, seed):
    """``run``'s outputs in float64 plain torch."""

    kind, train = case["kind"], case["train"]
    x = {k: (t if t.dtype is torch.bool else t.double()) for k, t in _inputs(case, seed).items()}
    if kind in ("triangle", "msa", "single"):
        if kind == "triangle":
            major = lambda t: t[0].transpose(1, 2).contiguous()  # noqa: E731  (rows, H, N, D)
        else:
            major = lambda t: t.contiguous()  # noqa: E731
        q, k, v = (major(x[name]) for name in ("query", "key", "value"))
        mask = x.get("mask")
        mask = mask[0] if mask is not None and kind == "triangle" else mask
        bias = x["bias"].reshape(x["bias"].shape[-3:])
        dout, dstage = None, []
        if kind == "single":
            att = _exact_attention(q, k, v, mask, bias, None)[0]
            stage = [att, x["single"], x["gate_weight"], x["output_weight"]]
            for t in stage:
                t.requires_grad_(train)
            out = _exact_gate(*stage)
            if not train:
                return out
            dout, *dstage = torch.autograd.grad(out, stage, x["dout"])
        elif train:
            dout = major(x["dout"])
        res = _exact_attention(q, k, v, mask, bias, dout)
        if kind == "triangle":
            res[:4] = [t.transpose(1, 2)[None] for t in res[:4]]
        if not train:
            return res[0]
        res[4] = res[4].reshape(x["bias"].shape)
        return (out.detach(), *res[1:], *dstage) if kind == "single" else tuple(res)
    leaves = _leaves(x)
    for t in leaves:
        t.requires_grad_(train)
    if kind == "gate":
        out = _exact_gate(x["attention"], x["single"], x["gate_weight"], x["output_weight"])
    elif kind == "trimul":
        out = _exact_trimul(x, case["direction"])
    else:
        out = torch.nn.functional.layer_norm(x["input"], (case["width"],), x["weight"], x["bias"])
    return (out.detach(), *torch.autograd.grad(out, leaves, x["dout"])) if train else out


# ----------------------------------------------------------------- tolerances


def tolerance(case):
    """About four times the largest 2-norm error of an output against the float64 reference, as measured: float32
    up to 7e-7; bfloat16 2.4e-3 in attention, 5.2e-3 where more roundings follow each other (gate, triangle
    multiplication), 1.7e-3 in LayerNorm; float16 an eighth of bfloat16."""

    if case["dtype"] == "f32":
        return {"rel": 3e-6}
    rel = {"triangle": 1e-2, "msa": 1e-2, "norm": 7e-3}.get(case["kind"], 2e-2)
    return {"rel": rel if case["dtype"] == "bf16" else rel / 8}
