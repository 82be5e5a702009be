"""The work that a user of this library has it do, as cases that can be timed and compared.

Four kinds of call cover what the path is for:

  gemv   a decode step's projections: one token times a Q4_K, Q6_K or Q8_0 matrix
  head   the LM head of a decode or draft-verify step: Q8_0 logits of 1..16 tokens and the top-64 row of each
  dense  a prompt's projections: many tokens times a Q4_K matrix, bf16 or f32 rows
  moe    one mixture-of-experts sublayer from its input rows to its output rows, composed as the host class composes it:
         router projection -> top-k -> routed experts -> shared expert -> shared router -> weighted sum,
         for one token (decode), 2..8 (draft verify) and 9..2048 (a prompt's chunk)

Weights are random bytes under the block scales that synth.py draws; everything is made on the GPU from the seed.
"""
import importlib
import math

import torch

capi = importlib.import_module("tokspur-public_amd.capi")

Q5_1, Q8_0, Q4_K, Q6_K = 7, 8, 12, 14
TYPES = {"q5_1": Q5_1, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
BLOCK = {Q5_1: (32, 24), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}  # weights, bytes

# (channels, hidden units, experts, selected) of the sublayers: the benchmark's, the engine's own, and two smaller models'
LAYERS = ((2048, 512, 512, 10), (2560, 640, 512, 10), (2048, 768, 128, 8), (1024, 512, 64, 4))


def listed():
    return [
        # decode: one projection of 2048 columns, the smallest call there is (4.7 MB of weights)
        {"name": "gemv_q4k_4096x2048", "op": "gemv", "type": "q4_k", "rows": 4096, "columns": 2048},
        # decode: the Q6_K matrices of a mixed file (value and down projections), an odd number of rows, 2560 columns
        {"name": "gemv_q6k_2731x2560", "op": "gemv", "type": "q6_k", "rows": 2731, "columns": 2560},
        # draft verify: four tokens' logits over the whole vocabulary
        {"name": "head_m4_151936x2048", "op": "head", "layout": "gguf", "tokens": 4, "vocabulary": 151936, "columns": 2048},
        # a short prompt in f32 rows, ragged tiles, the engine's width
        {"name": "dense_m37_6100x2560", "op": "dense", "tokens": 37, "rows": 6100, "columns": 2560, "bf16": False},
        # a middling prompt
        {"name": "dense_m450_8192x2560", "op": "dense", "tokens": 450, "rows": 8192, "columns": 2560, "bf16": True},
        # a long prompt's chunk
        {"name": "dense_m2048_8192x2048", "op": "dense", "tokens": 2048, "rows": 8192, "columns": 2048, "bf16": True},
        # decode: one token through the benchmark's sublayer
        {"name": "moe_t1_2048x512", "op": "moe", "tokens": 1, "channels": 2048, "hidden": 512, "experts": 512, "selected": 10, "down": "q6_k"},
        # draft verify: eight tokens through it
        {"name": "moe_t8_2048x512", "op": "moe", "tokens": 8, "channels": 2048, "hidden": 512, "experts": 512, "selected": 10, "down": "q6_k"},
        # draft verify on the engine's own experts and kinds
        {"name": "moe_t5_2560x640", "op": "moe", "tokens": 5, "channels": 2560, "hidden": 640, "experts": 512, "selected": 10, "down": "q8_0"},
        # a short prompt: every expert's weights for a handful of rows each
        {"name": "moe_t203_2048x512", "op": "moe", "tokens": 203, "channels": 2048, "hidden": 512, "experts": 512, "selected": 10, "down": "q6_k"},
        # a full chunk on the benchmark's experts, loads from a few to some hundred rows
        {"name": "moe_t2048_2048x512", "op": "moe", "tokens": 2048, "channels": 2048, "hidden": 512, "experts": 512, "selected": 10, "down": "q6_k"},
        # a full chunk on the engine's experts
        {"name": "moe_t2048_2560x640", "op": "moe", "tokens": 2048, "channels": 2560, "hidden": 640, "experts": 512, "selected": 10, "down": "q8_0"},
    ]


def _between(rng, low, high):
    """A whole number, even over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    op = rng.choice(("gemv", "head", "dense", "moe", "moe"))
    if op == "gemv":
        return {"op": "gemv", "type": rng.choice(("q4_k", "q6_k", "q8_0")), "rows": _between(rng, 512, 40000),
                "columns": 256 * _between(rng, 2, 24)}
    if op == "head":
        return {"op": "head", "layout": rng.choice(("gguf", "q8_lanes_v1")), "tokens": rng.randint(1, 16),
                "vocabulary": _between(rng, 32000, 151936), "columns": rng.choice((1024, 2048, 2560))}
    if op == "dense":
        return {"op": "dense", "tokens": _between(rng, 9, 2048), "rows": _between(rng, 512, 8192), "columns": 256 * rng.randint(2, 8) if rng.random() < 0.5 else 2560,
                "bf16": rng.random() < 0.5}
    channels, hidden, experts, selected = rng.choice(LAYERS)
    tokens = rng.randint(1, 8) if rng.random() < 0.5 else _between(rng, 9, 2048)
    downs = ("q6_k", "q8_0", "q5_1") if hidden % 256 == 0 else ("q8_0", "q5_1")
    return {"op": "moe", "tokens": tokens, "channels": channels, "hidden": hidden, "experts": experts, "selected": selected, "down": rng.choice(downs)}


# ------------------------------------------------------------------ inputs

class _Maker:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.gen, device="cuda") * scale

    def bytes(self, *shape, below=256):
        return torch.randint(0, below, shape, dtype=torch.uint8, device="cuda", generator=self.gen)

    def halves(self, *shape, scale, positive=True):
        v = self.normal(*shape, scale=scale)
        return (v.abs() if positive else v).half().view(torch.uint8)

    def quants(self, *shape):
        q = self.bytes(*shape)
        return q.masked_fill_(q == 128, 129)  # -128 is no Q8_0 code

    def rows(self, kind, rows, columns):
        """A matrix in GGUF rows."""
        per, size = BLOCK[kind]
        n = rows * columns // per
        out = self.quants(n, size) if kind == Q8_0 else self.bytes(n, size)
        if kind == Q8_0:
            out[:, 0:2] = self.halves(n, 1, scale=0.01)
        elif kind == Q4_K:
            out[:, 0:4] = self.halves(n, 2, scale=0.02)
        else:
            out[:, 208:210] = self.halves(n, 1, scale=0.02)
        return out.view(-1)

    def planes(self, kind, experts, rows, columns):
        """Experts in Pack v3 planes, [experts, bytes]."""
        spec = capi.make_expert_spec(kind, columns, rows)
        n = rows * spec.blocks_per_row
        if kind == Q8_0:
            out = self.quants(experts, spec.planar_expert_bytes)
            out[:, spec.dm_offset:] = self.halves(experts, n, scale=0.01)
        elif kind == Q5_1:
            out = self.bytes(experts, spec.planar_expert_bytes)
            out[:, spec.dm_offset:] = self.halves(experts, 2 * n, scale=0.02, positive=False)
        elif kind == Q4_K:
            out = self.bytes(experts, spec.planar_expert_bytes)
            out[:, spec.sm_offset:spec.dm_offset] &= 63
            out[:, spec.dm_offset:] = self.halves(experts, 2 * n, scale=0.02)
        else:
            out = self.bytes(experts, spec.planar_expert_bytes)
            out[:, spec.dm_offset:] = self.halves(experts, n, scale=0.02)
        return out


class _Experts(capi.PlanarMoeWeights):
    """A sublayer's experts, made in their planes as a Pack v3 file holds them."""

    def __init__(self, dev, make, down, channels, hidden, experts):
        self.gu_type, self.dn_type = Q4_K, down
        self.channels, self.hidden, self.experts = channels, hidden, experts
        self.gu_spec, self.dn_spec = capi.make_expert_spec(Q4_K, channels, hidden), capi.make_expert_spec(down, hidden, channels)
        self.pair_lo, self.pair_hi = make.planes(Q4_K, experts, hidden, channels).view(-1), make.planes(Q4_K, experts, hidden, channels).view(-1)
        self.down = make.planes(down, experts, channels, hidden).view(-1)
        self.union_meta = dev.zeros(2320, "int32")


class _SharedExpert(capi.PlanarSharedExpert):
    def __init__(self, make, channels, hidden):
        self.channels, self.hidden = channels, hidden
        self.gate, self.up = make.planes(Q4_K, 1, hidden, channels).view(-1), make.planes(Q4_K, 1, hidden, channels).view(-1)
        self.down = make.planes(Q6_K, 1, channels, hidden).view(-1)


def prepare(case, seed):
    dev, make = capi.Device(), _Maker(seed)
    s = {"case": case, "dev": dev}
    if case["op"] == "gemv":
        s.update(w=make.rows(TYPES[case["type"]], case["rows"], case["columns"]), x=make.normal(case["columns"]), y=dev.empty(case["rows"]))
    elif case["op"] == "head":
        tokens, vocabulary, columns = case["tokens"], case["vocabulary"], case["columns"]
        w = make.rows(Q8_0, vocabulary, columns)
        if case["layout"] == "q8_lanes_v1":  # scales first, then sixteen blocks at a time, their bytes of one index side by side
            blocks = w.view(vocabulary, columns // 32, 34)
            runs = blocks[:, :, 2:].reshape(vocabulary, columns // 512, 16, 32).transpose(2, 3)
            w = torch.cat((blocks[:, :, :2].reshape(vocabulary, -1), runs.reshape(vocabulary, -1)), dim=1).view(-1)
        s.update(w=w, x=make.normal(tokens, columns), y=dev.empty((tokens, vocabulary)), layout=capi.LAYOUT_GGUF if case["layout"] == "gguf" else capi.LAYOUT_Q8_LANES_V1,
                 scratch=dev.empty(capi.logit_topk_scratch_bytes(tokens, vocabulary), "uint8"), top=dev.empty(capi.logit_topk_output_bytes(tokens), "uint8"))
    elif case["op"] == "dense":
        tokens, rows, columns = case["tokens"], case["rows"], case["columns"]
        x = make.normal(tokens, columns)
        s.update(w=make.rows(Q4_K, rows, columns), x=x.bfloat16() if case["bf16"] else x, workspace=dev.empty(capi.dense_mm_workspace_bytes(tokens, columns), "uint8"),
                 y=dev.empty((tokens, rows), "bfloat16" if case["bf16"] else "float32"))
    else:
        tokens, channels, hidden, experts, selected, down = (case[k] for k in ("tokens", "channels", "hidden", "experts", "selected", "down"))
        # the router prefers some experts, by a Zipf law at a quarter of its strength: the first 64 channels carry an offset
        # that every token shares, and an expert's weights there its preference
        x = make.normal(tokens, channels)
        x[:, :64] += 1.0
        router = make.normal(experts, channels, scale=channels ** -0.5)
        rank = torch.randperm(experts, generator=make.gen, device="cuda") + 1
        router[:, :64] += (-0.275 / 64) * torch.log(rank.float())[:, None]
        s.update(x=x, router=router, shared_router=make.normal(1, channels, scale=channels ** -0.5), w=_Experts(dev, make, TYPES[down], channels, hidden, experts),
                 logits=dev.empty((tokens, experts)), ids=dev.zeros((tokens, selected), "int32"), weights=dev.zeros((tokens, selected)),
                 y=dev.empty((tokens * selected, channels)), shared_y=dev.empty((tokens, channels)), shared_logit=dev.empty(tokens), out=dev.empty((tokens, channels)))
        rides = down == "q6_k"  # the shared expert comes in the routed experts' formats and rides in their launches
        if rides:
            s.update(shared=_SharedExpert(make, channels, hidden))
        else:
            s.update(shared=None, shared_gate=make.rows(Q8_0, hidden, channels), shared_up=make.rows(Q8_0, hidden, channels), shared_down=make.rows(Q8_0, channels, hidden),
                     gate_rows=dev.empty((tokens, hidden)), up_rows=dev.empty((tokens, hidden)),
                     q8_workspace=dev.empty(max(capi.dense_mm_q8_workspace_bytes(tokens, channels, hidden), capi.dense_mm_q8_workspace_bytes(tokens, hidden, channels)), "uint8"))
        if tokens <= 8:
            s.update(h=dev.empty((tokens * selected, hidden)), shared_h=dev.empty((tokens, hidden)))
        else:
            s.update(scratch=capi.GroupedScratch(dev, tokens, selected, experts, channels, hidden, with_shared=rides))
    return s


# ------------------------------------------------------------------ one pass

def _dense_q8(s, matrix, x, columns, rows, out):
    """A shared expert's product: from 32 rows on the matrix is staged once, below that it is streamed past the rows."""
    tokens = s["case"]["tokens"]
    if tokens >= 32:
        return capi.dense_mm_q8_staged(s["dev"], capi.LAYOUT_GGUF, matrix, x, tokens, columns, rows, out=out, workspace=s["q8_workspace"])
    return capi.dense_mm_q8(s["dev"], capi.LAYOUT_GGUF, matrix, x, tokens, columns, rows, out=out)


def _moe(s):
    case, dev = s["case"], s["dev"]
    tokens, channels, hidden, experts, selected = case["tokens"], case["channels"], case["hidden"], case["experts"], case["selected"]
    if tokens == 1:
        dev.gemv(0, s["router"], s["x"], channels, experts, y=s["logits"])
    else:
        dev.router_f32_batch(s["router"], s["x"], tokens, channels, experts, out=s["logits"])
    dev.route(s["logits"], selected, 0, True, tokens=tokens, out=(s["ids"], s["weights"]))
    shared = {} if s["shared"] is None else {"shared": s["shared"], "shared_y": s["shared_y"]}
    if tokens <= 8:
        if shared:
            shared["shared_h"] = s["shared_h"]
        capi.planar_moe_routed_m8(dev, s["w"], s["ids"], s["x"], tokens, selected, h=s["h"], y=s["y"], **shared)
    else:
        capi.planar_nax_grouped_moe(dev, s["w"], s["ids"], s["x"], tokens, selected, s["scratch"], y=s["y"], **shared)
    if s["shared"] is None:
        _dense_q8(s, s["shared_gate"], s["x"], channels, hidden, s["gate_rows"])
        _dense_q8(s, s["shared_up"], s["x"], channels, hidden, s["up_rows"])
        dev.swiglu(s["gate_rows"], s["up_rows"], out=s["gate_rows"])
        _dense_q8(s, s["shared_down"], s["gate_rows"], hidden, channels, s["shared_y"])
    dev.gemv_rows(0, s["shared_router"], s["x"], s["shared_logit"], tokens, channels, 1, channels * 4, 4)
    dev.mixture(s["y"], s["weights"], s["shared_y"], s["shared_logit"], channels, selected, tokens=tokens, out=s["out"])
    return {"out": s["out"], "ids": s["ids"], "weights": s["weights"]}


def run(s):
    case, dev = s["case"], s["dev"]
    if case["op"] == "gemv":
        return dev.gemv(TYPES[case["type"]], s["w"], s["x"], case["columns"], case["rows"], y=s["y"])
    if case["op"] == "dense":
        tokens, rows, columns = case["tokens"], case["rows"], case["columns"]
        return capi.dense_mm(dev, Q4_K, capi.LAYOUT_GGUF, s["w"], s["x"], tokens, columns, rows, out=s["y"], out_bf16=case["bf16"], workspace=s["workspace"])
    if case["op"] == "head":
        tokens, vocabulary, columns = case["tokens"], case["vocabulary"], case["columns"]
        if tokens in (1, 2, 4, 8):
            dev.q8_matvec_many(s["w"], s["x"], columns, vocabulary, tokens, layout=s["layout"], y=s["y"])
        else:
            capi.dense_mm_q8(dev, s["layout"], s["w"], s["x"], tokens, columns, vocabulary, out=s["y"])
        capi.logit_topk(dev, s["y"], tokens, vocabulary, scratch=s["scratch"], out=s["top"])
        top = s["top"].view(torch.int32).view(tokens, 132)  # four counts, 64 ids, 64 values
        return {"logits": s["y"], "counts": top[:, :4], "ids": top[:, 4:68], "values": top[:, 68:].view(torch.float32)}
    return _moe(s)


# ------------------------------------------------------------------ what a pass cannot do without

def _matrix_bytes(kind, rows, columns):
    per, size = BLOCK[kind]
    return rows * columns // per * size


def work(case):
    if case["op"] == "gemv":
        r, c = case["rows"], case["columns"]
        return {"bytes": _matrix_bytes(TYPES[case["type"]], r, c) + 4 * (r + c), "flops": 2 * r * c}
    if case["op"] == "head":
        t, v, c = case["tokens"], case["vocabulary"], case["columns"]
        return {"bytes": _matrix_bytes(Q8_0, v, c) + t * (4 * c + 4 * v + 528), "flops": 2 * t * v * c}
    if case["op"] == "dense":
        t, r, c, item = case["tokens"], case["rows"], case["columns"], 2 if case["bf16"] else 4
        return {"bytes": _matrix_bytes(Q4_K, r, c) + t * (r + c) * item, "flops": 2 * t * r * c}
    t, c, h, e, k, down = (case[n] for n in ("tokens", "channels", "hidden", "experts", "selected", "down"))
    expert = _matrix_bytes(Q4_K, 2 * h, c) + _matrix_bytes(TYPES[down], c, h)
    shared = expert if down == "q6_k" else _matrix_bytes(Q8_0, 2 * h, c) + _matrix_bytes(Q8_0, c, h)
    met = e * (1 - (1 - k / e) ** t)  # distinct experts of t even draws of k
    return {"bytes": met * expert + shared + 4 * c * (e + 1) + t * (8 * c + 8 * k), "flops": 2 * t * c * (3 * h * (k + 1) + e + 1)}


def tolerance(case):
    if case["op"] == "gemv":
        return {"rel": 1e-5}  # f32 sums
    if case["op"] == "head":
        return {"rel": 1e-5, "differ": 0.01}  # f32 sums; near ties may change places in a row's ids
    if case["op"] == "dense":
        if case["bf16"]:
            return {"rel": 4e-3}  # the result's eight bits
        # f32 sums of exact products for few rows; from 512 rows on a weight is rounded once to half (the entry point's contract)
        return {"rel": 1e-3 if case["tokens"] >= 512 else 1e-5}
    # the rows between the two products, and the weights of the Q8_0 and Q5_1 planes, are halves
    return {"rel": 1e-3, "differ": 0.001}
