"""The work whose time matters: what a program that runs or finetunes an RWKV-7
model on packed weights has this package do, through its public entry points.

A block of width d has the projections r, k, v, o [d, d], the FFN key [4d, d]
and the FFN value [d, 4d]; the model widths are 768 (0.1B), 2048 (1.5B), 2560
(2.9B) and 4096 (7.2B) with a vocabulary of 65536.  The kinds of case:

  block       one block's six QuantizedLinear modules called one by one, with
              the QuantizedEmbedding lookup of the m tokens and the head on the
              last one where `vocab` is set: an eager decode step at small m,
              a prompt at larger m.
  decode      decode steps of `layers` blocks in dependency order through
              GroupedQmv handles kept by the program (r/k/v together, then o,
              key, value), and the head, for m sequences.
  sweep       every projection of `layers` blocks in one GroupedQmv.
  train       a QLoRA step of one block: LoRALinear over QuantizedLinear,
              forward and backward, gradients of x and of the adapters.
  sb6         the same on a `.rwkvq` (sb6) base: LoRALinear over the r/k/v/o
              bases, the FFN bases bare, as add_lora_rwkvq builds them.
  quantize    packing a bf16 or fp32 weight (model load, requantizing merge).
  dequantize  the dense form of a packed weight (adapter merge, export).

Weights are N(0, 0.02) quantized per group; activations are N(0, 1); incoming
gradients are N(0, 1e-2).
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "rwkv-metal_amd"))
import rwkvq  # noqa: E402

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
NAMES = ("r", "k", "v", "o", "key", "value")


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # an eager decode step of the smallest model, one sequence: launches and host work
        {"name": "block_0.1b_m1", "kind": "block", "d": 768, "vocab": 65536, "m": 1, "bits": 4,
         "gs": 64, "x": "bf16"},
        # generation with the 1.5B model, one sequence, fp32 residual stream (the default)
        {"name": "decode_1.5b_m1", "kind": "decode", "d": 2048, "vocab": 65536, "layers": 8,
         "m": 1, "bits": 4, "gs": 64, "x": "fp32"},
        # batched generation with the 2.9B model, an odd number of sequences in flight
        {"name": "decode_2.9b_m11", "kind": "decode", "d": 2560, "vocab": 65536, "layers": 4,
         "m": 11, "bits": 4, "gs": 64, "x": "bf16"},
        # the packed weights of a mixed-width 7.2B model's 3-bit body streamed once
        {"name": "sweep_7.2b_3bit_m1", "kind": "sweep", "d": 4096, "layers": 8, "m": 1, "bits": 3,
         "gs": 64, "x": "bf16"},
        # a short prompt (or the sequences of a larger decode batch) on the 1.5B model
        {"name": "prompt_1.5b_m77", "kind": "block", "d": 2048, "vocab": 65536, "m": 77, "bits": 4,
         "gs": 64, "x": "bf16"},
        # a prompt of ordinary length on the 2.9B model, fp32 residual stream
        {"name": "prompt_2.9b_m1000", "kind": "block", "d": 2560, "vocab": 65536, "m": 1000,
         "bits": 4, "gs": 64, "x": "fp32"},
        # a long prompt on the 7.2B model, 8-bit weights
        {"name": "prompt_7.2b_8bit_m2048", "kind": "block", "d": 4096, "vocab": 65536, "m": 2048,
         "bits": 8, "gs": 64, "x": "bf16"},
        # QLoRA finetuning of the 1.5B model, 8 sequences of 512 tokens
        {"name": "train_1.5b_m4096_r16", "kind": "train", "d": 2048, "m": 4096, "rank": 16,
         "bits": 4, "gs": 64, "x": "bf16"},
        # QLoRA on one short sequence, rank 32, fp32 residual stream
        {"name": "train_0.1b_m200_r32", "kind": "train", "d": 768, "m": 200, "rank": 32, "bits": 4,
         "gs": 64, "x": "fp32"},
        # QLoRA on the repacked sb6 base at B*T = 128
        {"name": "sb6_native_1.5b_m128", "kind": "sb6", "backend": "native", "d": 2048, "m": 128,
         "rank": 16, "xbits": 1, "x": "fp32"},
        # packing the largest weight, the 1.5B head
        {"name": "quantize_head_1.5b", "kind": "quantize", "rows": 65536, "cols": 2048, "bits": 4,
         "gs": 64, "w": "bf16"},
        # the dense form of a 2.9B FFN key at 6 bits
        {"name": "dequantize_2.9b_6bit", "kind": "dequantize", "rows": 10240, "cols": 2560,
         "bits": 6, "gs": 64, "s": "bf16"},
    ]


# what one drawn block may cost: the largest listed one's multiply-adds
MOST_MACS = 2048 * 12 * 4096 * 4096


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _width(rng, step, lo=512, hi=4096):
    return step * max(1, round(_log(rng, lo, hi) / step))


def draw(rng):
    kind = rng.choice(["block", "prompt", "prompt", "decode", "decode", "sweep", "train", "train",
                       "sb6", "quantize", "dequantize"])
    bits = rng.choice([4, 4, 4, 4, 8, 8, 3, 3, 6, 5, 2])
    gs = rng.choice([64, 64, 64, 128, 32])
    # most programs run the models' own widths, which are multiples of 256
    d = _width(rng, rng.choice([256, 256, max(64, gs)]))
    x = rng.choice(["bf16", "bf16", "fp32"])
    vocab = rng.choice([65536, 65536, 32000 + rng.randrange(9000)])
    if kind == "block":
        return {"kind": "block", "d": d, "vocab": vocab, "m": rng.randint(1, 16), "bits": bits,
                "gs": gs, "x": x}
    if kind == "prompt":
        m = round(_log(rng, 17, min(4096, MOST_MACS / (12 * d * d))))
        return {"kind": "block", "d": d, "vocab": vocab, "m": m, "bits": bits, "gs": gs, "x": x}
    if kind in ("decode", "sweep"):
        c = {"kind": kind, "d": d, "layers": rng.randint(2, 8 if kind == "sweep" or d < 2560 else 4),
             "m": rng.choice([1, 1, 2, 4, 8, rng.randint(1, 16)]), "bits": bits, "gs": gs, "x": x}
        if kind == "decode":
            c["vocab"] = vocab
        return c
    if kind == "train":
        m = round(_log(rng, 32, min(4096, MOST_MACS / 2 / (12 * d * d))))
        return {"kind": "train", "d": d, "m": m, "rank": rng.choice([16, 16, 32, 64, 8]),
                "bits": rng.choice([4, 4, 4, 8]), "gs": gs, "x": x}
    if kind == "sb6":
        m = round(_log(rng, 32, min(1024, MOST_MACS / 4 / (12 * d * d))))
        return {"kind": "sb6", "backend": rng.choice(["native", "native", "hybrid", "dense"]),
                "d": d, "m": m, "rank": 16, "xbits": rng.choice([0, 1, 2]), "x": x}
    rows = round(_log(rng, 300, 65536))
    cols = _width(rng, max(64, gs), 512, min(8192, 65536 * 2048 / rows))
    dt = rng.choice(["bf16", "bf16", "fp32"])
    return {"kind": kind, "rows": rows, "cols": cols, "bits": bits, "gs": gs,
            "w" if kind == "quantize" else "s": dt}


# ------------------------------------------------------------------- the data

def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEVICE) * std).to(dtype)


def _pack(codes, bits):
    """uint8 codes [R, K] -> int32 words [R, K*bits/32]: an LSB-first bitstream per row."""
    r, k = codes.shape
    c = codes.reshape(r, k // 32, 32)
    words = torch.zeros(r, k // 32, bits, dtype=torch.int64, device=codes.device)
    for j in range(32):
        w, off = divmod(j * bits, 32)
        v = c[:, :, j].to(torch.int64) << off
        words[:, :, w] |= v & 0xFFFFFFFF
        if off + bits > 32:
            words[:, :, w + 1] |= v >> 32
    return words.reshape(r, -1).to(torch.int32)


class Packed:
    """A weight [rows, cols] of N(0, 0.02) values in affine groups: its codes, scales, biases."""

    def __init__(self, g, rows, cols, bits, gs, dtype=torch.bfloat16):
        self.rows, self.cols, self.bits, self.gs = rows, cols, bits, gs
        w = _randn(g, rows, cols // gs, gs, std=0.02)
        lo, hi = w.amin(-1), w.amax(-1)
        self.scales = ((hi - lo) / (2 ** bits - 1)).to(dtype)
        self.biases = lo.to(dtype)
        q = (w - self.biases.float()[..., None]) / self.scales.float()[..., None]
        self.codes = q.round_().clamp_(0, 2 ** bits - 1).to(torch.uint8).reshape(rows, cols)

    def packed(self):
        return _pack(self.codes, self.bits), self.scales, self.biases

    def linear(self):
        q = rwkvq.QuantizedLinear(self.cols, self.rows, False, self.gs, self.bits, device=DEVICE,
                                  dtype=self.scales.dtype)
        q.weight, q.scales, q.biases = self.packed()
        return q

    def embedding(self):
        q = rwkvq.QuantizedEmbedding(self.rows, self.cols, self.gs, self.bits, device=DEVICE,
                                     dtype=self.scales.dtype)
        q.weight, q.scales, q.biases = self.packed()
        return q

    def rows64(self, at=slice(None)):
        """The weight's rows in 64 bits."""
        q = self.codes[at].double().reshape(-1, self.cols // self.gs, self.gs)
        w = q * self.scales[at].double()[..., None] + self.biases[at].double()[..., None]
        return w.reshape(-1, self.cols)


class Sb6:
    """A weight [rows, cols] of N(0, 0.02) values in sb6 blocks of 32 codes of 4 + xbits bits."""

    def __init__(self, g, rows, cols, xbits):
        self.shape, self.xbits, nb = (rows, cols), xbits, cols // 32
        self.sb = next(n for n in (8, 4, 2, 1) if nb % n == 0)
        w = _randn(g, rows, nb, 32, std=0.02)
        lo, hi = w.amin(-1), w.amax(-1)
        top = 2 ** (4 + xbits) - 1
        sup = (rows, nb // self.sb, self.sb)
        d = (((hi - lo) / top).reshape(sup).amax(-1) / 63).half()
        dm = (lo.reshape(sup).abs().amax(-1) / -31).half()
        over = lambda t: t.float().repeat_interleave(self.sb, 1)  # noqa: E731
        qs = ((hi - lo) / top / over(d)).round().clamp(1, 63)
        qm = (lo / over(dm)).round().clamp(-31, 32)
        self.scale, self.low = (qs * over(d)).half().float(), (qm * over(dm)).half().float()
        q = (w - self.low[..., None]) / self.scale[..., None]
        self.codes = q.round_().clamp_(0, top).to(torch.uint8)
        c = self.codes
        parts = [(c[..., :16] & 15) | ((c[..., 16:] & 15) << 4)]
        for x in range(xbits):
            bit = (c >> (4 + x)) & 1
            parts.append(torch.stack([sum(bit[..., 8 * b + i] << i for i in range(8))
                                      for b in range(4)], -1).to(torch.uint8))
        self.qblk = torch.cat(parts, -1).reshape(rows, -1)
        self.qsqm = torch.stack([qs.to(torch.uint8), qm.to(torch.int8).view(torch.uint8)],
                                -1).reshape(rows, -1)
        self.ddm = torch.stack([d, dm], -1).reshape(rows, -1)

    def base(self, backend):
        lin = rwkvq.RwkvqLinear(self.qblk, self.qsqm, self.ddm, self.shape, 32, self.sb, self.xbits)
        return {"native": rwkvq.RwkvqNativeLinear, "hybrid": rwkvq.RwkvqHybridLinear,
                "dense": lambda x: x}[backend](lin)

    def rows64(self):
        w = self.codes.double() * self.scale.double()[..., None] + self.low.double()[..., None]
        return w.reshape(self.shape)


def _shapes(d):
    return [(d, d)] * 4 + [(4 * d, d), (d, 4 * d)]


def _data(case, seed):
    """Everything random in a case, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    xdt = DTYPES[case.get("x", "bf16")]
    if kind == "quantize":
        return {"w": _randn(g, case["rows"], case["cols"], std=0.02, dtype=DTYPES[case["w"]])}
    if kind == "dequantize":
        return {"w": Packed(g, case["rows"], case["cols"], case["bits"], case["gs"],
                            DTYPES[case["s"]])}
    d, m = case["d"], case["m"]
    if kind in ("decode", "sweep"):
        ws, xs = [], []
        for _ in range(case["layers"]):
            xs.append([_randn(g, m, k, dtype=xdt) for k in (d, d, d, 4 * d)])
            ws.append([Packed(g, r, k, case["bits"], case["gs"]) for r, k in _shapes(d)])
        out = {"w": ws, "x": xs}
        if kind == "decode":
            out["head"] = Packed(g, case["vocab"], d, case["bits"], case["gs"])
            out["xh"] = _randn(g, m, d, dtype=xdt)
        return out
    if kind == "block":
        out = {"w": [Packed(g, r, k, case["bits"], case["gs"]) for r, k in _shapes(d)],
               "x": [_randn(g, 1, m, k, dtype=xdt) for k in (d, d, d, 4 * d)]}
        if case["vocab"]:
            # the embedding shares the head's shape; its lookups read m rows of it
            out["head"] = Packed(g, case["vocab"], d, case["bits"], case["gs"])
            out["idx"] = torch.randint(case["vocab"], (1, m), generator=g, device=DEVICE)
        return out
    if kind == "train":
        ws = [Packed(g, r, k, case["bits"], case["gs"]) for r, k in _shapes(d)]
    else:
        ws = [Sb6(g, r, k, case["xbits"]) for r, k in _shapes(d)]
    rank = case["rank"]
    return {"w": ws,
            "x": [_randn(g, m, k, dtype=xdt) for k in (d, d, d, 4 * d)],
            "dy": [_randn(g, m, r, std=1e-2, dtype=xdt) for r, _ in _shapes(d)],
            "a": [_randn(g, rank, k, std=k ** -0.5, dtype=torch.bfloat16) for _, k in _shapes(d)],
            "b": [_randn(g, r, rank, std=0.01, dtype=torch.bfloat16) for r, _ in _shapes(d)]}


#: which of a block's inputs each projection reads (r/k/v, o, key, value)
READS = (0, 0, 0, 1, 2, 3)


def _adapted(case):
    return range(6) if case["kind"] == "train" else range(4)


def _alpha(case):
    return 2.0 * case["rank"]


# ---------------------------------------------------------------- the program

def prepare(case, seed):
    t, kind = _data(case, seed), case["kind"]
    if kind == "quantize":
        return {"case": case, "w": t["w"]}
    if kind == "dequantize":
        return {"case": case, "w": t["w"].packed()}
    if kind in ("decode", "sweep"):
        groups = []
        every = [([x[0], x[0], x[0]], ws[:3]) for x, ws in zip(t["x"], t["w"])]
        for i, (x, ws) in enumerate(zip(t["x"], t["w"])):
            levels = [every[i], ([x[1]], [ws[3]]), ([x[2]], [ws[4]]), ([x[3]], [ws[5]])]
            groups += levels
        if kind == "sweep":
            groups = [(sum((xs for xs, _ in groups), []), sum((ws for _, ws in groups), []))]
        else:
            groups.append(([t["xh"]], [t["head"]]))
        handles = [rwkvq.GroupedQmv(xs, [w.packed() for w in ws], case["gs"], case["bits"])
                   for xs, ws in groups]
        return {"case": case, "handles": handles}
    if kind == "block":
        s = {"case": case, "x": t["x"], "layers": [w.linear() for w in t["w"]]}
        if case["vocab"]:
            s["idx"], s["head"], s["emb"] = t["idx"], t["head"].linear(), t["head"].embedding()
        return s
    layers = []
    for i, w in enumerate(t["w"]):
        base = w.linear() if kind == "train" else w.base(case["backend"])
        if i in _adapted(case):
            base = rwkvq.LoRALinear(rank=case["rank"], alpha=_alpha(case), base_module=base)
            with torch.no_grad():
                base.lora_a.copy_(t["a"][i])
                base.lora_b.copy_(t["b"][i])
        layers.append(base)
    xs = [t["x"][j].clone().requires_grad_(True) for j in READS]
    params = xs + [p for i in _adapted(case) for p in (layers[i].lora_a, layers[i].lora_b)]
    return {"case": case, "layers": layers, "x": xs, "dy": t["dy"], "params": params}


def run(state):
    kind = state["case"]["kind"]
    if kind == "quantize":
        return rwkvq.quantize(state["w"], state["case"]["gs"], state["case"]["bits"])
    if kind == "dequantize":
        return rwkvq.dequantize(*state["w"], state["case"]["gs"], state["case"]["bits"])
    if kind in ("decode", "sweep"):
        return [h.run() for h in state["handles"]]
    if kind == "block":
        with torch.no_grad():
            x, out = state["x"], []
            if "emb" in state:
                out.append(state["emb"](state["idx"]))
            out += [layer(x[j]) for layer, j in zip(state["layers"], READS)]
            if "head" in state:
                out.append(state["head"](x[0][:, -1:]))
        return out
    ys = [layer(x) for layer, x in zip(state["layers"], state["x"])]
    grads = torch.autograd.grad(ys, state["params"], state["dy"])
    return {"y": [y.detach() for y in ys], "grads": list(grads)}


def exact(case, seed):
    t, kind = _data(case, seed), case["kind"]
    if kind == "quantize":
        w = t["w"].double().reshape(case["rows"], -1, case["gs"])
        lo, hi = w.amin(-1), w.amax(-1)
        down = lo.abs() > hi.abs()
        scale = ((hi - lo) / (2 ** case["bits"] - 1)).clamp_min(1e-7)
        scale = torch.where(down, scale, -scale)
        edge = torch.where(down, lo, hi)
        q0 = (edge / scale).round()
        scale = torch.where(q0 != 0, edge / q0, scale)
        return None, scale, torch.where(q0 != 0, edge, torch.zeros_like(edge))
    if kind == "dequantize":
        return t["w"].rows64()
    if kind in ("decode", "sweep"):
        every = [[x[j].double() @ w.rows64().t() for w, j in zip(ws, READS)]
                 for x, ws in zip(t["x"], t["w"])]
        if kind == "sweep":
            return [sum(every, [])]
        out = []
        for ys in every:
            out += [ys[:3], ys[3:4], ys[4:5], ys[5:6]]
        return out + [[t["xh"].double() @ t["head"].rows64().t()]]
    if kind == "block":
        out = []
        if case["vocab"]:
            out.append(t["head"].rows64(t["idx"].reshape(-1)).reshape(1, case["m"], case["d"]))
        out += [t["x"][j].double() @ w.rows64().t() for w, j in zip(t["w"], READS)]
        if case["vocab"]:
            out.append(t["x"][0][:, -1:].double() @ t["head"].rows64().t())
        return out
    ys, dxs, grads = [], [], []
    for i, w in enumerate(t["w"]):
        x, dy, full = t["x"][READS[i]].double(), t["dy"][i].double(), w.rows64()
        if i in _adapted(case):
            a, b, s = t["a"][i].double(), t["b"][i].double(), _alpha(case) / case["rank"]
            full = full + s * (b @ a)
            grads += [s * ((dy @ b).t() @ x), s * (dy.t() @ (x @ a.t()))]
        ys.append(x @ full.t())
        dxs.append(dy @ full)
    return {"y": ys, "grads": dxs + grads}


# ------------------------------------------------------------ what it must do

def _size(name):
    return 2 if name == "bf16" else 4


def _packed_bytes(rows, cols, bits, gs, size=2):
    return rows * cols * bits // 8 + 2 * rows * (cols // gs) * size


def work(case):
    kind = case["kind"]
    if kind in ("quantize", "dequantize"):
        r, k, size = case["rows"], case["cols"], _size(case.get("w") or case.get("s"))
        return {"bytes": r * k * size + _packed_bytes(r, k, case["bits"], case["gs"], size),
                "flops": 2 * r * k}
    d, m, xs = case["d"], case["m"], _size(case["x"])
    shapes = _shapes(d)
    macs = m * sum(r * k for r, k in shapes)
    acts = m * sum({j: shapes[i][1] for i, j in enumerate(READS)}.values()) * xs
    outs = m * sum(r for r, _ in shapes) * xs
    if kind in ("block", "decode", "sweep"):
        weights = sum(_packed_bytes(r, k, case["bits"], case["gs"]) for r, k in shapes)
        n = case.get("layers", 1)
        total, flops = n * (weights + acts + outs), 2 * n * macs
        if case.get("vocab"):
            hm = m if kind == "decode" else 1
            total += _packed_bytes(case["vocab"], d, case["bits"], case["gs"])
            total += hm * case["vocab"] * xs + (m * d * xs if kind == "decode" else 0)
            flops += 2 * hm * case["vocab"] * d
            if kind == "block":  # the embedding's m rows, and their dense form
                total += _packed_bytes(m, d, case["bits"], case["gs"]) + m * d * 2 + m * 8
        return {"bytes": total, "flops": flops}
    if kind == "train":
        weights = sum(_packed_bytes(r, k, case["bits"], case["gs"]) for r, k in shapes)
    else:
        weights = sum(r * k * (4 + case["xbits"]) // 8 + r * (k // 32) * 2 + r * (k // 256) * 4
                      for r, k in shapes)
    dx = m * sum(k for _, k in shapes) * xs
    adapted = [shapes[i] for i in _adapted(case)]
    low = sum(r + k for r, k in adapted) * case["rank"]
    # x, dy read; y, dx written; adapters read, their gradients written
    return {"bytes": weights + 2 * outs + 2 * dx + 2 * low * 2,
            "flops": 4 * macs + 2 * m * low * 4}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "dequantize"):
        return "exact"
    # About four times the error against exact() (which is in turn the size of
    # the difference between two correct implementations).
    if kind in ("decode", "sweep"):
        # codes, scales and biases enter exactly; fp32 x keeps 16 bits or more
        # at m <= 2 (3e-6), else x or y is rounded to bf16 (1.7e-3)
        return {"rel": 1.2e-5 if case["x"] == "fp32" and case["m"] <= 2 else 7e-3}
    if kind == "block":
        # as decode at m <= 16; beyond, the weights are rounded to bf16 too
        # (2.3e-3)
        return {"rel": 7e-3 if case["m"] <= 16 else 1e-2}
    # bf16 weights, bf16 z and u between the low-rank products, bf16 gradients
    # of the adapters (2.3e-3 to 3.3e-3)
    return {"rel": 1.2e-2}
