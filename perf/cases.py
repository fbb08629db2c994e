"""The work a program gives this backend, as cases that can be timed and checked.

Every case goes through a public entry point: one projection
(zg_gemv_device, zg_gemv_device_fused), one Gated DeltaNet layer's decode step
or chunked prefill, one attention layer's decode step, the resident decode
step of a session, and the batched prefill of a prompt.  Widths are those of
the 2B-shaped and the 0.8B-shaped model (hidden 2048 / FFN 6144 and hidden
1024 / FFN 3584, 16 GDN heads of 128, 8 query and 2 KV heads of 256,
vocabulary 151936).  Weights are random blocks of the named codec.

`exact` restates each path in float64 torch: weights dequantised exactly,
activations coded where the codec's rule codes them (Q8_0), K and V rounded
to the cache type, everything else in 64 bits.
"""
import math

import numpy as np
import torch

from zerogravity_amd import _lib as L
from zerogravity_amd import chunk, qwen35
from zerogravity_amd import regions as R

CODEC = {"q8_0": 8, "q4_k": 12}
BYTES = {"q8_0": 34 / 32, "q4_k": 144 / 256}
VOCAB = 151936
HEADS, DIM = 16, 128          # Gated DeltaNet
QH, KVH, HD = 8, 2, 256       # attention
THETA = 1e7 ** (-2.0 / 64.0)  # RoPE over the first 64 dimensions
EPS = 1e-6
WIDTHS = {1024: 3584, 2048: 6144}  # hidden -> FFN
DEV = "cuda"


def listed():
    return [
        # one request decoding: its FFN gate/up with the norm before and the
        # SwiGLU after it, the smallest call a program makes per layer
        dict(name="gate_up_1row", kind="fused", form="rms_glu", codec="q4_k", rows=1, columns=2048, outputs=12288),
        # the LM head of a small batch on the codec of the published Q8_0 checkpoints
        dict(name="head_q8_11rows", kind="projection", codec="q8_0", rows=11, columns=2048, outputs=VOCAB, norm=True),
        # a prompt's largest projection, and a short ragged prompt's FFN down
        dict(name="prompt_gate_up_2048", kind="projection", codec="q4_k", rows=2048, columns=2048, outputs=12288,
             norm=True),
        dict(name="prompt_down_601", kind="projection", codec="q4_k", rows=601, columns=6144, outputs=2048,
             norm=False),
        # one GDN layer and one attention layer of a continuous batch, a token each
        dict(name="gdn_step_32rows", kind="gdn_step", rows=32, heads=16),
        dict(name="attention_step_8rows", kind="attention_step", rows=8, context=3001, kv="bf16", form="split"),
        # one GDN layer over a prompt
        dict(name="gdn_prefill_2048", kind="gdn_prefill", tokens=2048, heads=16),
        # the whole resident decode step: one request; blocks of the schedule
        # for a few requests, a full batch, and the Q8_0 model
        dict(name="decode_1row", kind="decode", codec="q4_k", hidden=2048, layers=24, rows=1, prefix=2048, kv="bf16"),
        dict(name="decode_3rows", kind="decode", codec="q4_k", hidden=2048, layers=8, rows=3, prefix=1500, kv="bf16"),
        dict(name="decode_32rows", kind="decode", codec="q4_k", hidden=2048, layers=8, rows=32, prefix=2048,
             kv="bf16"),
        dict(name="decode_q8_1row", kind="decode", codec="q8_0", hidden=1024, layers=8, rows=1, prefix=1024,
             kv="bf16"),
        # admission of a request: the whole model over its prompt, logits to the host
        dict(name="prefill_2048", kind="prefill", codec="q4_k", hidden=2048, layers=24, tokens=2048, kv="bf16"),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["fused", "projection", "prompt", "gdn_step", "attention_step", "gdn_prefill", "decode",
                       "decode", "prefill"])
    if kind == "fused":
        form = rng.choice(["rms_glu", "rms_store", "plain_residual"])
        return dict(kind=kind, form=form, codec="q4_k", rows=rng.randint(1, 4),
                    columns=rng.choice([1024, 2048] if form == "rms_glu" else [1024, 2048, 3584, 6144]),
                    outputs=2 * log(128, 8192) if form == "rms_glu" else log(256, 16384))
    if kind == "projection":
        return dict(kind=kind, codec=rng.choice(["q4_k", "q8_0"]), rows=log(1, 64),
                    columns=rng.choice([1024, 2048, 3584, 6144]), outputs=log(256, 16384), norm=rng.random() < 0.5)
    if kind == "prompt":
        return dict(kind="projection", codec="q4_k", rows=log(65, 4096), columns=rng.choice([1024, 2048, 3584, 6144]),
                    outputs=log(512, 16384), norm=rng.random() < 0.5)
    if kind == "gdn_step":
        return dict(kind=kind, rows=log(1, 64), heads=rng.choice([16, 16, 32]))
    if kind == "attention_step":
        rows = log(1, 64)
        return dict(kind=kind, rows=rows, context=log(16, min(8192, 131072 // rows)), kv=rng.choice(["bf16", "f32"]),
                    form=rng.choice(["split", "split", "exact"]))
    if kind == "gdn_prefill":
        return dict(kind=kind, tokens=log(1, 8192), heads=16)
    hidden = rng.choice([1024, 2048])
    if kind == "decode":
        rows = log(1, 64)
        return dict(kind=kind, codec=rng.choice(["q4_k", "q4_k", "q8_0"]), hidden=hidden, layers=4, rows=rows,
                    prefix=log(16, min(4096, 65536 // rows)), kv=rng.choice(["bf16", "bf16", "f32"]))
    return dict(kind="prefill", codec="q4_k", hidden=hidden, layers=4, tokens=log(17, 8192), kv="bf16")


# ------------------------------------------------------------------- inputs

class Source:
    """Random inputs on the GPU, made from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, scale=1.0, mean=0.0):
        return mean + scale * torch.randn(*shape, device=DEV, generator=self.g)

    def uniform(self, n, lo, hi):
        return lo + (hi - lo) * torch.rand(n, device=DEV, generator=self.g)

    def below(self, hi, *shape):
        return torch.randint(0, hi, shape, device=DEV, generator=self.g)

    def matrix(self, codec, rows, cols):
        """[rows * blocks, block bytes] uint8, outputs about the input's size."""
        if codec == "q4_k":
            n = rows * (cols // 256)
            b = torch.randint(0, 256, (n, 144), device=DEV, generator=self.g, dtype=torch.uint8)
            d = self.uniform(n, 0.5, 1.5) / (258.0 * math.sqrt(cols))
            b[:, 0:2] = d.half().view(torch.uint8).view(n, 2)
            b[:, 2:4] = (d * 7.5 * self.uniform(n, 0.8, 1.2)).half().view(torch.uint8).view(n, 2)
            return b
        n = rows * (cols // 32)
        b = torch.randint(-127, 128, (n, 34), device=DEV, generator=self.g, dtype=torch.int8).view(torch.uint8)
        d = self.uniform(n, 0.5, 1.5) * (1.7 / (127.0 * math.sqrt(cols)))
        b[:, 0:2] = d.half().view(torch.uint8).view(n, 2)
        return b


def host(t):
    return t.reshape(-1).cpu().numpy()


def geometry(case):
    return dict(hidden=case["hidden"], layers=case["layers"], ffn=WIDTHS[case["hidden"]], vocab=VOCAB,
                gdn_heads=HEADS, gdn_dim=DIM, q_heads=QH, kv_heads=KVH, head_dim=HD, full_attention_interval=4,
                max_context=262144, eps=EPS)


def is_full(i):
    return (i + 1) % 4 == 0


def model_tensors(case, src):
    """{GGUF name: (codec or None, columns, rows, GPU tensor)} in load order."""
    h, f, w = case["hidden"], WIDTHS[case["hidden"]], HEADS * DIM
    t = {}

    def mat(name, k, n):
        t[name] = (case["codec"], k, n, src.matrix(case["codec"], n, k))

    def vec(name, v, k=None, n=1):
        t[name] = (None, k or v.numel(), n, v)

    mat("token_embd.weight", h, VOCAB)
    vec("output_norm.weight", src.normal(h, scale=0.1, mean=1.0))
    for i in range(case["layers"]):
        p = f"blk.{i}."
        vec(p + "attn_norm.weight", src.normal(h, scale=0.1, mean=1.0))
        vec(p + "post_attention_norm.weight", src.normal(h, scale=0.1, mean=1.0))
        mat(p + "ffn_gate.weight", h, f)
        mat(p + "ffn_up.weight", h, f)
        mat(p + "ffn_down.weight", f, h)
        if is_full(i):
            mat(p + "attn_q.weight", h, 2 * QH * HD)
            mat(p + "attn_k.weight", h, KVH * HD)
            mat(p + "attn_v.weight", h, KVH * HD)
            mat(p + "attn_output.weight", QH * HD, h)
            vec(p + "attn_q_norm.weight", src.normal(HD, scale=0.1, mean=1.0))
            vec(p + "attn_k_norm.weight", src.normal(HD, scale=0.1, mean=1.0))
        else:
            mat(p + "attn_qkv.weight", h, 3 * w)
            mat(p + "attn_gate.weight", h, w)
            mat(p + "ssm_alpha.weight", h, HEADS)
            mat(p + "ssm_beta.weight", h, HEADS)
            mat(p + "ssm_out.weight", w, h)
            vec(p + "ssm_conv1d.weight", src.normal(3 * w, 4, scale=0.5), 4, 3 * w)
            vec(p + "ssm_norm.weight", src.normal(DIM, scale=0.1, mean=1.0))
            vec(p + "ssm_a", -torch.exp(src.normal(HEADS, scale=0.5)))
            vec(p + "ssm_dt.bias", src.normal(HEADS))
    return t


def load_model(case, tensors):
    table = {n: (CODEC[c] if c else 0, k, rows, host(v.contiguous().view(torch.uint8)))
             for n, (c, k, rows, v) in tensors.items()}
    return qwen35.QwenModelHip(geometry(case), table)


def row_states(case, src):
    """Up to four prompts' states, ragged in length: (tokens, per layer the
    conv history [3W, 3] and state [H, 128, 128], or keys and values
    [tokens, 512]).  A batch's other rows are forks of them."""
    out = []
    for r in range(min(case["rows"], 4)):
        n = case["prefix"] - r * (case["prefix"] // 8)
        layers = []
        for i in range(case["layers"]):
            if is_full(i):
                layers.append((src.normal(n, KVH * HD), src.normal(n, KVH * HD)))
            else:
                layers.append((src.normal(3 * HEADS * DIM, 3, scale=0.5), src.normal(HEADS, DIM, DIM, scale=0.02)))
        out.append((n, layers))
    return out


def attention_inputs(case, src):
    rows, t = case["rows"], case["context"]
    dtype = torch.bfloat16 if case["kv"] == "bf16" else torch.float32
    return dict(proj=src.normal(rows, (2 * QH + 2 * KVH) * HD), q_norm=src.normal(HD, scale=0.1, mean=1.0),
                k_norm=src.normal(HD, scale=0.1, mean=1.0),
                positions=(t - 1 - src.below(t // 4 + 1, rows)).int(),
                keys=src.normal(rows, t, KVH * HD).to(dtype), values=src.normal(rows, t, KVH * HD).to(dtype))


def gdn_step_inputs(case, src):
    rows, h = case["rows"], case["heads"]
    w = h * DIM
    return dict(proj=src.normal(rows, 4 * w + 2 * h), conv_w=src.normal(3 * w, 4, scale=0.5),
                ring=src.normal(rows, 3 * w, 4, scale=0.5), positions=(4 + src.below(4096, rows)).int(),
                dt=src.normal(h, scale=0.1), a=-torch.exp(src.normal(h)),
                state=src.normal(rows, h, DIM, DIM, scale=0.02))


def gdn_prefill_inputs(case, src):
    n, h = case["tokens"], case["heads"]
    q, k, v = (src.normal(n, h, DIM).bfloat16().float() for _ in range(3))
    beta = torch.sigmoid(src.normal(n, h)).bfloat16().float()
    decay = -torch.nn.functional.softplus(src.normal(n, h)) * torch.exp(src.normal(n, h, scale=0.5))
    return dict(q=q, k=k, v=v, beta=beta, decay=decay.clamp(max=0.0), state=src.normal(h, DIM, DIM, scale=0.02))


def projection_inputs(case, src):
    k, n, m = case["columns"], case["outputs"], case["rows"]
    return dict(weight=src.matrix(case["codec"], n, k), x=src.normal(m, k), gamma=src.normal(k, scale=0.1, mean=1.0),
                y=src.normal(m, n // 2 if case.get("form") == "rms_glu" else n))


STREAMS = []


def one_stream():
    """A program decodes on one stream: each pass follows the one before."""
    if not STREAMS:
        STREAMS.append(torch.cuda.Stream())
    return STREAMS[0]


ROOM = 1024  # decode steps a session holds past its prompt before the rows return to it


def prepare(case, seed):
    src = Source(seed)
    kind = case["kind"]
    s = dict(case=case, lib=L.lib(), stream=one_stream())
    s["s"] = s["stream"].cuda_stream
    if kind in ("fused", "projection"):
        s.update(projection_inputs(case, src), kern=R.HipMatVecKernel(0))
        s["ctx"] = s["kern"].ctx
        s["w"] = s["kern"].register(1 + seed, "w", CODEC[case["codec"]], case["columns"], case["outputs"],
                                    host(s.pop("weight")))
        if kind == "projection":
            # the weight as a serving program holds it: a first call lays it out
            torch.cuda.synchronize()
            run(s)
    elif kind == "gdn_step":
        s.update(gdn_step_inputs(case, src), ctx=L.Context(0))
        s["core"] = torch.empty(case["rows"], case["heads"] * DIM, device=DEV)
    elif kind == "attention_step":
        s.update(attention_inputs(case, src), ctx=L.Context(0))
        rows, t = case["rows"], case["context"]
        size = (s["lib"].zg_attn_decode_split_workspace_bytes(rows, QH, KVH, t) if case["form"] == "split" else
                s["lib"].zg_attn_decode_workspace_bytes(rows, QH, t))
        s["workspace"] = torch.empty(size, dtype=torch.uint8, device=DEV)
        s["out"] = torch.empty(rows, QH * HD, device=DEV)
    elif kind == "gdn_prefill":
        s.update(gdn_prefill_inputs(case, src), ctx=L.Context(0))
        s["out"] = torch.empty(case["tokens"], case["heads"], DIM, device=DEV)
        s["start"], s["state"] = s["state"], torch.empty_like(s["state"])
    elif kind == "decode":
        rows = case["rows"]
        s["model"] = load_model(case, model_tensors(case, src))
        s["ctx"] = s["model"].ctx
        s["session"] = s["model"].session(rows, case["prefix"] + ROOM, L.BF16 if case["kv"] == "bf16" else L.F32)
        s["snapshots"] = []
        for r, (n, layers) in enumerate(row_states(case, src)):
            image = torch.cat([t.reshape(-1) for pair in layers for t in pair])
            s["session"].load_state(host(image), n, r)
            s["snapshots"].append(s["session"].snapshot(r))
        s["tokens"] = src.below(VOCAB, rows).int()
        s["greedy"] = torch.empty(rows, dtype=torch.int32, device=DEV)
        s["logits"] = torch.empty(rows, VOCAB, device=DEV)
        s["left"] = 0
        rewind(s)
    else:
        s["model"] = load_model(case, model_tensors(case, src))
        s["session"] = s["model"].session(1, case["tokens"], L.BF16 if case["kv"] == "bf16" else L.F32)
        s["tokens"] = src.below(VOCAB, case["tokens"]).cpu().numpy().astype(np.uint32)
    torch.cuda.synchronize()
    return s


def rewind(s):
    """Every row back to the prompt it forks (a request starting over)."""
    for r in range(s["case"]["rows"]):
        s["session"].restore(s["snapshots"][r % len(s["snapshots"])], r)
    s["left"] = ROOM


def p(t):
    return t.data_ptr()


def run(s):
    case, lib, kind = s["case"], s["lib"], s["case"]["kind"]
    if kind == "projection":
        s["ctx"].check(lib.zg_gemv_device(s["ctx"].h, s["w"].h, p(s["x"]), L.F32, case["rows"],
                                          p(s["gamma"]) if case["norm"] else None, EPS, p(s["y"]), s["s"]))
        return s["y"]
    if kind == "fused":
        rms, glu = case["form"] != "plain_residual", case["form"] == "rms_glu"
        s["ctx"].check(lib.zg_gemv_device_fused(
            s["ctx"].h, s["w"].h, case["rows"], 0 if rms else 3,
            {"rms_glu": 2, "rms_store": 0, "plain_residual": 1}[case["form"]], p(s["x"]), case["columns"], None, 0,
            p(s["gamma"]) if rms else None, EPS, DIM, p(s["y"]), case["outputs"] // 2 if glu else case["outputs"],
            None, None, None, None, s["s"]))
        return s["y"]
    if kind == "gdn_step":
        h = case["heads"]
        s["ctx"].check(lib.zg_gdn_decode_device(s["ctx"].h, case["rows"], h, p(s["proj"]), (4 * DIM + 2) * h,
                                                p(s["conv_w"]), p(s["ring"]), p(s["positions"]), p(s["dt"]),
                                                p(s["a"]), EPS, p(s["state"]), p(s["core"]), s["s"]))
        return {"core": s["core"], "state": s["state"], "ring": s["ring"]}
    if kind == "attention_step":
        call = lib.zg_attn_decode_split_device if case["form"] == "split" else lib.zg_attn_decode_device
        s["ctx"].check(call(s["ctx"].h, case["rows"], QH, KVH, p(s["proj"]), (2 * QH + 2 * KVH) * HD, p(s["q_norm"]),
                            p(s["k_norm"]), EPS, THETA, p(s["positions"]), p(s["keys"]), p(s["values"]),
                            case["context"], L.BF16 if case["kv"] == "bf16" else L.F32, p(s["workspace"]),
                            p(s["out"]), s["s"]))
        return {"out": s["out"], "keys": s["keys"], "values": s["values"]}
    if kind == "gdn_prefill":
        with torch.cuda.stream(s["stream"]):
            s["state"].copy_(s["start"])
        chunk.prefill_device(s["ctx"], case["tokens"], case["heads"], s["q"], s["k"], s["v"], s["beta"], s["decay"],
                             s["state"], s["out"], s["s"])
        return {"out": s["out"], "state": s["state"]}
    if kind == "decode":
        if s["left"] == 0:
            rewind(s)
        s["left"] -= 1
        s["ctx"].check(lib.zg_decode_step_device(s["session"].h, case["rows"], p(s["tokens"]), p(s["logits"]),
                                                 p(s["greedy"]), s["s"]))
        return s["logits"]
    s["session"].reset_row(0)
    return s["session"].prefill_batched(s["tokens"])


# --------------------------------------------------------- work, tolerances

def chunk_flops(tokens, heads):
    """One chunk of 64 tokens of one head: A and intra, the two unit-lower
    solves, W S and dq S, intra corr, dk^T corr."""
    c, d = 64, DIM
    return 2 * -(-tokens // c) * heads * (2 * c * c * d + c * (c - 1) * d + 3 * c * d * d + c * c * d)


def layer_weights(hidden):
    """Weight elements of (a GDN layer, an attention layer)."""
    f, w = WIDTHS[hidden], HEADS * DIM
    return (hidden * (4 * w + 2 * HEADS) + w * hidden + 3 * hidden * f,
            hidden * (2 * QH + 2 * KVH) * HD + QH * HD * hidden + 3 * hidden * f)


def work(case):
    kind = case["kind"]
    if kind in ("fused", "projection"):
        m, k, n = case["rows"], case["columns"], case["outputs"]
        glu, resid = case.get("form") == "rms_glu", case.get("form") == "plain_residual"
        return dict(bytes=n * k * BYTES[case["codec"]] + 4 * m * (k + (n // 2 if glu else n) * (2 if resid else 1)),
                    flops=2 * m * n * k)
    if kind == "gdn_step":
        b, h = case["rows"], case["heads"]
        w = h * DIM
        return dict(bytes=4 * (b * (2 * h * DIM * DIM + 4 * w + 2 * h + w + 3 * w * 4) + 3 * w * 4),
                    flops=b * h * 7 * DIM * DIM)
    if kind == "attention_step":
        cached = case["rows"] * case["context"] * 7 // 8  # the mean position
        return dict(bytes=cached * 2 * KVH * HD * (2 if case["kv"] == "bf16" else 4)
                    + case["rows"] * 4 * (3 * QH + 2 * KVH) * HD, flops=cached * 4 * QH * HD)
    if kind == "gdn_prefill":
        n, h = case["tokens"], case["heads"]
        return dict(bytes=4 * (n * h * (4 * DIM + 2) + 2 * h * DIM * DIM), flops=chunk_flops(n, h))
    n_attn = case["layers"] // 4
    n_gdn = case["layers"] - n_attn
    gdn, attn = layer_weights(case["hidden"])
    params = n_gdn * gdn + n_attn * attn
    head = VOCAB * case["hidden"]
    if kind == "decode":
        rows = case["rows"]
        mean = sum(case["prefix"] - r % 4 * (case["prefix"] // 8) for r in range(rows))  # cached tokens, all rows
        state = n_gdn * 4 * (2 * HEADS * DIM * DIM + 3 * HEADS * DIM * 4)
        kv = n_attn * mean * 2 * KVH * HD * (2 if case["kv"] == "bf16" else 4)
        return dict(bytes=(params + head) * BYTES[case["codec"]] + rows * (state + 4 * VOCAB) + kv,
                    flops=2 * rows * (params + head) + n_attn * mean * 4 * QH * HD)
    n = case["tokens"]
    return dict(bytes=(params + head) * BYTES[case["codec"]] + n_attn * n * 2 * KVH * HD * 2
                + n_gdn * 8 * HEADS * DIM * DIM + 4 * VOCAB,
                flops=2 * n * params + 2 * head + n_gdn * chunk_flops(n, HEADS) + n_attn * 2 * n * (n + 1) * QH * HD)


def tolerance(case):
    """About four times the error measured against float64."""
    kind = case["kind"]
    if kind in ("fused", "projection"):
        # Q8_0: integer dots, 32-bit sums (1.5e-7).  Q4_K: f16 weights and
        # activations (4.4e-4), one row 16-bit activation codes (3e-5)
        return {"rel": 1e-5 if case["codec"] == "q8_0" else 2e-3}
    if kind in ("gdn_step", "gdn_prefill"):
        return {"rel": 1e-5}  # 32-bit sums (2e-7; over a prompt 2e-6)
    if kind == "attention_step":
        return {"rel": 3e-5}  # 32-bit sums and exponentials (6.5e-6)
    # Q4_K: the projections' 4e-4 through the layers (1.2e-3).  Q8_0: 1e-7,
    # or, once a rounding moves one activation code by one, the coding's own
    # step through the layers after it (1.7e-2)
    return {"rel": 5e-3 if case["codec"] == "q4_k" else 2.5e-2}


# -------------------------------------------------------------------- exact

def dequantize(codec, raw, rows, cols):
    """[rows, cols] float64."""
    b = raw.reshape(-1, raw.shape[-1])
    n = b.shape[0]
    half = lambda t: t.contiguous().view(torch.float16).double().view(n, 1)  # noqa: E731
    if codec == "q8_0":
        return (half(b[:, 0:2]) * b[:, 2:].view(torch.int8).double()).view(rows, cols)
    d, dmin, s, v = half(b[:, 0:2]), half(b[:, 2:4]), b[:, 4:16].int(), b[:, 16:144]
    out = torch.empty(n, 256, dtype=torch.float64, device=b.device)
    for g in range(8):
        if g < 4:
            sc, mn = s[:, g] & 63, s[:, g + 4] & 63
        else:
            sc = (s[:, g + 4] & 15) | ((s[:, g - 4] >> 6) << 4)
            mn = (s[:, g + 4] >> 4) | ((s[:, g] >> 6) << 4)
        q = v[:, 32 * (g // 2):32 * (g // 2) + 32]
        q = (q >> 4) if g % 2 else (q & 15)
        out[:, 32 * g:32 * g + 32] = d * sc.view(n, 1) * q.double() - dmin * mn.view(n, 1)
    return out.view(rows, cols)


def code_q8(x):
    """The codec's dynamic activation coding: per 32 values, codes in
    [-128, 127] of the largest magnitude / 127, that scale rounded to f16."""
    b = x.reshape(-1, 32)
    top = b.abs().amax(1, keepdim=True)
    codes = torch.round(b * torch.where(top > 0, 127.0 / top, top)).clamp(-128, 127)
    return (codes * (top / 127.0).half().double()).view_as(x)


def multiply(codec, raw, rows, cols, x):
    """x [m, cols] float64 times the packed [rows, cols] matrix, transposed."""
    x = code_q8(x) if codec == "q8_0" else x
    per, step = raw.shape[0] // rows, 16384
    return torch.cat([x @ dequantize(codec, raw[r * per:min(rows, r + step) * per], min(rows, r + step) - r,
                                     cols).t().contiguous() for r in range(0, rows, step)], 1)


def rms(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def silu(x):
    return x * torch.sigmoid(x)


def unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + EPS)


def delta_rule(q, k, v, gain, beta, s):
    """Token by token over dim 1 of [rows, n, heads, ...]; s [rows, heads, value, key]."""
    out = torch.empty_like(v)
    q, k = unit(q) / math.sqrt(DIM), unit(k)
    for t in range(q.shape[1]):
        s = s * gain[:, t, :, None, None]
        kt = k[:, t].unsqueeze(-1)
        corr = beta[:, t].unsqueeze(-1) * (v[:, t] - (s @ kt).squeeze(-1))
        s = s + corr.unsqueeze(-1) * k[:, t].unsqueeze(-2)
        out[:, t] = (s @ q[:, t].unsqueeze(-1)).squeeze(-1)
    return out, s


def rotate(x, pos):
    """x [n, heads, 256], pos [n]."""
    angle = pos.double().view(-1, 1, 1) * THETA ** torch.arange(32, dtype=torch.float64, device=x.device)
    c, s = torch.cos(angle), torch.sin(angle)
    a, b = x[..., :32], x[..., 32:64]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., 64:]], -1)


def attend(proj, q_norm, k_norm, pos, keys, values, dtype):
    """One row: proj [n, ...] of tokens at positions pos..pos+n-1 over the
    cached [pos, 512] keys and values (float64); the gated output [n, 2048]
    and the grown caches."""
    n = proj.shape[0]
    qg = proj[:, :2 * QH * HD].view(n, QH, 2, HD)
    at = torch.arange(pos, pos + n, device=proj.device)
    q = rotate(rms(qg[:, :, 0], q_norm), at)
    k = rotate(rms(proj[:, 2 * QH * HD:(2 * QH + KVH) * HD].view(n, KVH, HD), k_norm), at)
    v = proj[:, (2 * QH + KVH) * HD:]
    keys = torch.cat([keys, k.reshape(n, KVH * HD).float().to(dtype).double()])
    values = torch.cat([values, v.float().to(dtype).double()])
    late = torch.arange(pos + n, device=proj.device).view(1, -1) > at.view(-1, 1)
    out = torch.empty(n, QH, HD, dtype=torch.float64, device=proj.device)
    for h in range(QH):
        g = h // (QH // KVH)
        score = q[:, h] @ keys[:, g * HD:(g + 1) * HD].t().contiguous() / 16.0
        out[:, h] = torch.softmax(score.masked_fill(late, -math.inf), 1) @ values[:, g * HD:(g + 1) * HD]
    return (out * torch.sigmoid(qg[:, :, 1])).view(n, QH * HD), keys, values


def forward(case, t, tokens, positions, states, dtype):
    """tokens [rows, n] after `positions` cached tokens; logits of each row's last."""
    rows, n = tokens.shape
    hidden, w = case["hidden"], HEADS * DIM

    def mul(name, x):
        codec, k, outs, raw = t[name]
        return multiply(codec, raw, outs, k, x)

    codec, k, _, raw = t["token_embd.weight"]
    raw = raw.view(VOCAB, -1, raw.shape[-1])
    x = dequantize(codec, raw[tokens.reshape(-1)].reshape(-1, raw.shape[-1]), rows * n, k)
    for i in range(case["layers"]):
        b = f"blk.{i}."
        vec = lambda name: t[b + name][3].double()  # noqa: E731
        h = rms(x, vec("attn_norm.weight"))
        if is_full(i):
            proj = torch.cat([mul(b + f"attn_{m}.weight", h) for m in "qkv"], 1).view(rows, n, -1)
            mixed = torch.cat([attend(proj[r], vec("attn_q_norm.weight"), vec("attn_k_norm.weight"), positions[r],
                                      states[r][i][0].to(dtype).double(), states[r][i][1].to(dtype).double(),
                                      dtype)[0] for r in range(rows)])
            x = x + mul(b + "attn_output.weight", mixed)
        else:
            qkv = mul(b + "attn_qkv.weight", h).view(rows, n, 3 * w)
            past = torch.stack([states[r][i][0].double() for r in range(rows)])  # [rows, 3W, 3]
            seq = torch.cat([past.transpose(1, 2), qkv], 1)
            taps = vec("ssm_conv1d.weight").view(3 * w, 4)
            conv = silu(sum(seq[:, j:j + n] * taps[:, j] for j in range(4)))
            q, k, v = (conv[..., j * w:(j + 1) * w].reshape(rows, n, HEADS, DIM) for j in range(3))
            step = torch.nn.functional.softplus(mul(b + "ssm_alpha.weight", h) + vec("ssm_dt.bias"))
            gain = torch.exp(step * vec("ssm_a")).view(rows, n, HEADS)
            beta = torch.sigmoid(mul(b + "ssm_beta.weight", h)).view(rows, n, HEADS)
            core, _ = delta_rule(q, k, v, gain, beta, torch.stack([states[r][i][1].double() for r in range(rows)]))
            mixed = rms(core, vec("ssm_norm.weight")).view(rows * n, w) * silu(mul(b + "attn_gate.weight", h))
            x = x + mul(b + "ssm_out.weight", mixed)
        h = rms(x, vec("post_attention_norm.weight"))
        x = x + mul(b + "ffn_down.weight", silu(mul(b + "ffn_gate.weight", h)) * mul(b + "ffn_up.weight", h))
    last = x.view(rows, n, hidden)[:, -1]
    return mul("token_embd.weight", rms(last, t["output_norm.weight"][3]))


def exact(case, seed):
    src = Source(seed)
    kind = case["kind"]
    dtype = torch.bfloat16 if case.get("kv") == "bf16" else torch.float32
    if kind in ("fused", "projection"):
        i = projection_inputs(case, src)
        form = case.get("form")
        x = i["x"].double()
        if case.get("norm") or form in ("rms_glu", "rms_store"):
            x = rms(x, i["gamma"])
        y = multiply(case["codec"], i["weight"], case["outputs"], case["columns"], x)
        if form == "rms_glu":
            return y[:, case["outputs"] // 2:] * silu(y[:, :case["outputs"] // 2])
        return y + i["y"].double() if form == "plain_residual" else y
    if kind == "gdn_step":
        i = gdn_step_inputs(case, src)
        rows, h = case["rows"], case["heads"]
        w = h * DIM
        proj = i["proj"].double()
        slot = i["positions"].long() % 4
        ring = i["ring"].double()
        ring[torch.arange(rows, device=DEV), :, slot] = proj[:, :3 * w]
        order = (slot.view(-1, 1) + 1 + torch.arange(4, device=DEV)) % 4  # oldest to newest
        seq = torch.gather(ring, 2, order.view(rows, 1, 4).expand(rows, 3 * w, 4))
        conv = silu((seq * i["conv_w"].double()).sum(2))
        q, k, v = (conv[:, j * w:(j + 1) * w].reshape(rows, 1, h, DIM) for j in range(3))
        gain = torch.exp(torch.nn.functional.softplus(proj[:, 4 * w:4 * w + h] + i["dt"].double()) * i["a"].double())
        core, state = delta_rule(q, k, v, gain.view(rows, 1, h), torch.sigmoid(proj[:, 4 * w + h:]).view(rows, 1, h),
                                 i["state"].double())
        return {"core": core.reshape(rows, w), "state": state, "ring": ring}
    if kind == "attention_step":
        i = attention_inputs(case, src)
        keys, values, out = i["keys"].double(), i["values"].double(), []
        for r in range(case["rows"]):
            at = int(i["positions"][r])
            o, k, v = attend(i["proj"][r:r + 1].double(), i["q_norm"], i["k_norm"], at, keys[r, :at], values[r, :at],
                             dtype)
            out.append(o)
            keys[r, at], values[r, at] = k[-1], v[-1]
        return {"out": torch.cat(out), "keys": keys, "values": values}
    if kind == "gdn_prefill":
        i = {n: t.double().unsqueeze(0) for n, t in gdn_prefill_inputs(case, src).items()}
        out, state = delta_rule(i["q"], i["k"], i["v"], torch.exp(i["decay"]), i["beta"], i["state"])
        return {"out": out[0], "state": state[0]}
    t = model_tensors(case, src)
    if kind == "decode":
        prompts = row_states(case, src)
        rows = [prompts[r % len(prompts)] for r in range(case["rows"])]
        tokens = src.below(VOCAB, case["rows"]).view(-1, 1)
        return forward(case, t, tokens, [n for n, _ in rows], [s for _, s in rows], dtype)
    none = torch.zeros(0, KVH * HD, device=DEV)
    zero = [(none, none) if is_full(i) else (torch.zeros(3 * HEADS * DIM, 3, device=DEV),
                                             torch.zeros(HEADS, DIM, DIM, device=DEV)) for i in range(case["layers"])]
    return forward(case, t, src.below(VOCAB, case["tokens"]).view(1, -1), [0], [zero], dtype)[0]
