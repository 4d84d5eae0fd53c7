"""The work that programs give this backend, as measurable cases.

A program either drives a whole model (HipModel over gh_model_*: prefill of a prompt, then decode
steps) or, as the engine behind the trait boundary does, records single operations of each layer
into an encoder and submits them together (HipBackend over the gh_* operations). Both are here,
over the range of sizes the framework accepts: prompts and chunks of 1 to 2048 tokens, contexts up
to 32768, both weight formats, every GQA group, the 8B and 14B widths and arbitrary ones.

Model cases use a few blocks of the width in question (one case uses the whole 8B-shaped depth), so
that their outputs stay comparable and their states small; layer cases run over several layers'
weights or caches, as a forward pass does, so that no pass finds its data in a cache.
"""
import ctypes as C
import math

import numpy as np
import torch

from graph_horizon_amd import HipBackend, HipModel, synth
from graph_horizon_amd import _ffi as F

D8, FFN8 = 4096, 12288    # the 8B-shaped width
D14, FFN14 = 5120, 16384  # the 14B-shaped width
HEAD_DIM = 128
Q4K, Q6K = "q4_k", "q6_k"
FORMATS = {Q4K: F.FMT_Q4_K, Q6K: F.FMT_Q6_K}
BLOCK_BYTES = {Q4K: 144, Q6K: 210}
# Q4_K_M: V, down and output are Q6_K
LAYER = (("q", F.T_ATTN_Q, Q4K), ("k", F.T_ATTN_K, Q4K), ("v", F.T_ATTN_V, Q6K),
         ("o", F.T_ATTN_OUTPUT, Q4K), ("gate", F.T_FFN_GATE, Q4K), ("up", F.T_FFN_UP, Q4K),
         ("down", F.T_FFN_DOWN, Q6K))


def model_case(kind, d, ffn, blocks, vocab, n, base, kv_heads=8, group=4):
    return {"kind": kind, "d": d, "ffn": ffn, "blocks": blocks, "vocab": vocab, "n": n, "base": base,
            "kv_heads": kv_heads, "group": group}


def gemm_case(fmt, in_dim, out_dim, n, layers):
    return {"kind": "gemm", "fmt": fmt, "in_dim": in_dim, "out_dim": out_dim, "n": n, "layers": layers}


def attn_case(kind, n, base, layers, kv_heads=8, group=4):
    return {"kind": kind, "n": n, "base": base, "layers": layers, "kv_heads": kv_heads, "group": group}


def glue_case(d, ffn, rows, base, kv_heads=8, group=4):
    return {"kind": "glue", "d": d, "ffn": ffn, "n": rows, "base": base, "kv_heads": kv_heads, "group": group}


def listed():
    cases = {
        # the candidates of one sampled token (temperature with top-k), after every decode step
        "topk_40": {"kind": "topk", "vocab": 131072, "k": 40},
        # one token of greedy decode: the whole 8B-shaped model in a chat of ordinary length
        "decode_8b_520": model_case("decode", D8, FFN8, 34, 131072, 1, 520),
        # one token deep into a long document, 14B-shaped blocks
        "decode_14b_8000": model_case("decode", D14, FFN14, 8, 8192, 1, 8000),
        # a handful of new tokens in a conversation that is already in the cache (also what a
        # speculative decoder verifies at once)
        "prefill_8b_5": model_case("prefill", D8, FFN8, 4, 8192, 5, 300),
        # a short prompt
        "prefill_8b_100": model_case("prefill", D8, FFN8, 4, 8192, 100, 0),
        # a follow-up of some paragraphs on the larger model
        "prefill_14b_500": model_case("prefill", D14, FFN14, 4, 8192, 500, 700),
        # a full chunk of a long prompt
        "prefill_8b_2048": model_case("prefill", D8, FFN8, 4, 8192, 2048, 0),
        # one projection of a ragged batch, recorded op by op (the engine's matmul_batched)
        "gemm_down_300": gemm_case(Q6K, FFN8, D8, 300, 4),
        # the attention of one token over a full 32K cache
        "attn_decode_32k": attn_case("attn_decode", 1, 32767, 4),
        # the last chunk of an 8K prompt
        "attn_prefill_8k": attn_case("attn_prefill", 2048, 6144, 2),
        # eight query heads per kv head (64 heads over 8), a ragged chunk
        "attn_prefill_g8": attn_case("attn_prefill", 500, 300, 2, group=8),
        # the operations between the projections for a chunk, recorded op by op
        "glue_2000": glue_case(D8, FFN8, 2000, 0),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    heads = {"kv_heads": rng.choice((8, 8, 8, 4, 2)), "group": rng.choice((4, 4, 4, 8, 2, 1))}
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "prefill", "gemm", "gemm", "attn_decode",
                       "attn_prefill", "attn_prefill", "glue", "topk"))
    if kind == "topk":
        return {"kind": kind, "vocab": log_int(rng, 2000, 131072), "k": rng.randint(1, 128)}
    if kind == "gemm":
        return gemm_case(rng.choice((Q4K, Q6K)), 256 * rng.randint(4, 64), log_int(rng, 500, 16384),
                         log_int(rng, 1, 2048), rng.randint(1, 4))
    if kind == "attn_decode":
        return attn_case(kind, 1, log_int(rng, 1, 32767), rng.randint(1, 4), **heads)
    if kind == "attn_prefill":
        return attn_case(kind, log_int(rng, 8, 2048), rng.choice((0, log_int(rng, 1, 6144))), rng.randint(1, 2),
                         **heads)
    d, ffn = rng.choice(((D8, FFN8), (D14, FFN14), (256 * rng.randint(4, 20), 256 * rng.randint(8, 64))))
    if kind == "glue":
        return glue_case(d, ffn, log_int(rng, 1, 2048), rng.choice((0, log_int(rng, 1, 8000))), **heads)
    blocks, vocab = rng.randint(1, 4), log_int(rng, 2000, 32768)
    if kind == "decode":
        return model_case(kind, d, ffn, blocks, vocab, 1, log_int(rng, 1, 16000), **heads)
    case = model_case(kind, d, ffn, blocks, vocab, log_int(rng, 2, 2048), rng.choice((0, log_int(rng, 1, 4096))),
                      **heads)
    # no more work than a full chunk over four 8B-shaped blocks
    most = work(model_case(kind, D8, FFN8, 4, 8192, 2048, 0))["flops"]
    while work(case)["flops"] > most:
        case["n"] = case["n"] * 3 // 4
    return case


# ---- sizes and work ----

def dims(c):
    """(in, out) of each of a block's matrices."""
    qw, kw = c["kv_heads"] * c["group"] * HEAD_DIM, c["kv_heads"] * HEAD_DIM
    d, ffn = c["d"], c["ffn"]
    return {"q": (d, qw), "k": (d, kw), "v": (d, kw), "o": (qw, d), "gate": (d, ffn), "up": (d, ffn),
            "down": (ffn, d)}


def weight_bytes(fmt, in_dim, out_dim):
    return in_dim // 256 * BLOCK_BYTES[fmt] * out_dim


def attention_work(c, n, base, layers):
    """(bytes, flops) of causal attention over the cache: visible K and V once, Q in, the output out."""
    heads = c["kv_heads"] * c["group"]
    seen = n * base + n * (n + 1) // 2
    return (layers * (2 * (base + n) * c["kv_heads"] + 2 * n * heads) * HEAD_DIM * 2,
            layers * 4 * heads * HEAD_DIM * seen)


def work(case):
    c = case
    if c["kind"] == "topk":
        return {"bytes": 4 * c["vocab"] + 8 * c["k"], "flops": 0}
    if c["kind"] == "gemm":
        return {"bytes": c["layers"] * (weight_bytes(c["fmt"], c["in_dim"], c["out_dim"]) + 2 * c["n"] * c["out_dim"])
                + 2 * c["n"] * c["in_dim"], "flops": 2 * c["layers"] * c["n"] * c["in_dim"] * c["out_dim"]}
    if c["kind"].startswith("attn"):
        b, f = attention_work(c, c["n"], c["base"], c["layers"])
        return {"bytes": b, "flops": f}
    if c["kind"] == "glue":
        kw, qw = c["kv_heads"] * HEAD_DIM, c["kv_heads"] * c["group"] * HEAD_DIM
        # norm: x, out; RoPE: q and k in and out; append: k and v in and out; SiLU: two in, one
        # out; residual: x in and out, y
        per_row = 6 * c["d"] + 4 * (qw + kw) + 8 * kw + 6 * c["ffn"] + 10 * c["d"]
        return {"bytes": c["n"] * per_row, "flops": 0}
    mats = [(weight_bytes(fmt, *dims(c)[name]), dims(c)[name]) for name, _, fmt in LAYER]
    b, f = attention_work(c, c["n"], c["base"], c["blocks"])
    b += c["blocks"] * sum(w for w, _ in mats) + weight_bytes(Q6K, c["d"], c["vocab"]) + 4 * c["vocab"]
    f += 2 * c["n"] * c["blocks"] * sum(i * o for _, (i, o) in mats) + 2 * c["d"] * c["vocab"]
    return {"bytes": b, "flops": f}


# ---- states ----

_backend = None


def backend():
    """The program's one backend."""
    global _backend
    if _backend is None:
        _backend = HipBackend(0)
    return _backend


def handle(t):
    """A buffer handle over a tensor's memory."""
    return F.GhBuf(t.data_ptr(), t.numel() * t.element_size(), F.FMT_F16, F.BUF_VIEW, 0, 0)


class Model(HipModel):
    """A model that is given back with its last user."""

    def __del__(self):
        self.close()


class Memory:
    """A tensor's view of FP16 device memory that `owner` holds (a model, for its cache)."""

    def __init__(self, owner, addr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f2", "data": (addr, False), "version": 2}


class State:
    """What the program holds: buffers, weights and, for model cases, the model and its cache."""

    def __init__(self, case):
        self.case, self.weights = case, []

    def __del__(self):
        for w in self.weights:
            backend().free_buffer(w)


def generator(seed):
    g = torch.Generator("cuda")
    g.manual_seed(seed)
    return g


def normal(g, *shape, dtype=torch.float16):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def blocks_of(g, fmt, rows, in_dim, gain=1.0):
    """GGUF blocks [rows * in_dim / 256][bytes] of weights around 0 with a root mean square of about
    gain / sqrt(in_dim), which keeps activations of unit scale there. Q4_K: uniform quants and 6-bit
    scales, each sub-block's least weight about -7.5 of its steps, as quantizing a centred weight
    gives it; Q6_K: uniform quants, int8 N(0, 16) sub-block scales."""
    nb = rows * (in_dim // 256)
    size = BLOCK_BYTES[fmt]
    words = torch.randint(-2**31, 2**31, ((nb * size + 3) // 4,), generator=g, device="cuda", dtype=torch.int32)
    blk = words.view(torch.uint8)[:nb * size].view(nb, size)
    d = normal(g, nb, 1, dtype=torch.float32).abs() * (gain / ((168 if fmt == Q4K else 296) * math.sqrt(in_dim)))
    if fmt == Q4K:
        least = 7.5 * d * (1 + 0.05 * normal(g, nb, 1, dtype=torch.float32))
        blk[:, :4] = torch.cat([d, least], 1).half().view(torch.uint8)
        blk[:, 8:12] = blk[:, 4:8]  # the sub-blocks' minima equal to their scales
        blk[:, 12:16] = (blk[:, 12:16] & 15) * 17
    else:
        sc = normal(g, nb, 16, dtype=torch.float32).mul(16).round().clamp(-128, 127).to(torch.int8)
        blk[:, 192:208] = sc.view(torch.uint8)
        blk[:, 208:210] = d.half().view(torch.uint8)
    return blk


def host(t):
    return t.reshape(-1).cpu().numpy()


def model_inputs(c, seed):
    """The tensors of a model case in loading order, then its cache contents and tokens."""
    g = generator(seed)

    def norm_weight():
        return 1.0 + 0.05 * normal(g, c["d"], dtype=torch.float32)

    yield F.NO_LAYER, F.T_TOKEN_EMBD, Q4K, blocks_of(g, Q4K, c["vocab"], c["d"], math.sqrt(c["d"]))
    yield F.NO_LAYER, F.T_OUTPUT_NORM, None, norm_weight()
    yield F.NO_LAYER, F.T_OUTPUT, Q6K, blocks_of(g, Q6K, c["vocab"], c["d"])
    for li in range(c["blocks"]):
        yield li, F.T_ATTN_NORM, None, norm_weight()
        yield li, F.T_FFN_NORM, None, norm_weight()
        for name, tid, fmt in LAYER:
            i, o = dims(c)[name]
            yield li, tid, fmt, blocks_of(g, fmt, o, i)
        # what earlier calls left in this layer's cache
        yield li, "cache", None, (normal(g, c["base"], c["kv_heads"], HEAD_DIM),
                                  normal(g, c["base"], c["kv_heads"], HEAD_DIM))
    yield F.NO_LAYER, "tokens", None, torch.randint(0, c["vocab"], (c["n"],), generator=g, device="cuda")


def prepare_model(s, c, seed):
    hip = backend()
    context = c["base"] + c["n"] + 8
    shape = synth.Shape("case", c["blocks"], c["d"], c["ffn"], head_count=c["kv_heads"] * c["group"],
                        kv_head_count=c["kv_heads"], vocab_size=c["vocab"])
    s.model = Model(hip, synth.model_config(shape, context))
    kv = s.model.kv()
    whole = (c["blocks"], context, c["kv_heads"], HEAD_DIM)
    s.k, s.v = (torch.as_tensor(Memory(s.model, b.addr, whole), device="cuda") for b in (kv.k, kv.v))
    s.k.zero_()
    s.v.zero_()
    for li, tid, fmt, data in model_inputs(c, seed):
        if tid == "cache":
            s.k[li, :c["base"]], s.v[li, :c["base"]] = data
        elif tid == "tokens":
            s.tokens = data.cpu().numpy().astype(np.uint32)
        else:
            s.model.load_tensor(li, tid, FORMATS[fmt] if fmt else F.FMT_F32, host(data))


def kv_handle(k, v, c, layers, context):
    return F.GhKv(handle(k), handle(v), F.KV_F16, layers, context, c["kv_heads"], HEAD_DIM, HEAD_DIM)


def attn_inputs(c, seed):
    g = generator(seed)
    context = c["base"] + c["n"]
    cache = (c["layers"], context, c["kv_heads"], HEAD_DIM)
    return normal(g, *cache), normal(g, *cache), normal(g, c["layers"], c["n"], c["kv_heads"] * c["group"], HEAD_DIM)


def gemm_inputs(c, seed):
    g = generator(seed)
    yield normal(g, c["n"], c["in_dim"])
    for _ in range(c["layers"]):
        yield blocks_of(g, c["fmt"], c["out_dim"], c["in_dim"])


def glue_inputs(c, seed):
    g = generator(seed)
    n, heads = c["n"], c["kv_heads"] * c["group"]
    return {"x": normal(g, n, c["d"], dtype=torch.float32), "w": (1.0 + 0.05 * normal(g, c["d"], dtype=torch.float32)).half(),
            "q": normal(g, n, heads, HEAD_DIM), "k": normal(g, n, c["kv_heads"], HEAD_DIM),
            "v": normal(g, n, c["kv_heads"], HEAD_DIM), "gate": normal(g, n, c["ffn"]), "up": normal(g, n, c["ffn"]),
            "y": normal(g, n, c["d"])}


def topk_inputs(c, seed):
    return 3.0 * normal(generator(seed), c["vocab"], dtype=torch.float32)


def yarn_of():
    """The model family's RoPE parameters (synth.yarn_params): theta 1e6, YaRN factor 16 over 16384."""
    return dict(rope_dim=HEAD_DIM, original_context=16384, freq_base=1e6, factor=16.0, beta_fast=32.0, beta_slow=1.0,
                log_multiplier=1.0, q_temperature_scale=0.1)


def prepare(case, seed):
    c, hip = case, backend()
    s = State(c)
    if c["kind"] in ("decode", "prefill"):
        prepare_model(s, c, seed)
    elif c["kind"] == "gemm":
        data = gemm_inputs(c, seed)
        s.x = next(data)
        s.weights = [hip.load_weight(FORMATS[c["fmt"]], host(b), c["in_dim"], c["out_dim"]) for b in data]
        s.out = torch.empty(c["layers"], c["n"], c["out_dim"], dtype=torch.float16, device="cuda")
        s.bufs = (handle(s.x), [handle(o) for o in s.out])
    elif c["kind"].startswith("attn"):
        s.k, s.v, s.q = attn_inputs(c, seed)
        s.out = torch.empty_like(s.q)
        s.kv = kv_handle(s.k, s.v, c, c["layers"], c["base"] + c["n"])
        s.bufs = ([handle(o) for o in s.out], [handle(q) for q in s.q])
    elif c["kind"] == "glue":
        for name, t in glue_inputs(c, seed).items():
            setattr(s, name, t)
        s.normed, s.act = torch.empty_like(s.y), torch.empty_like(s.up)
        s.kc, s.vc = (torch.zeros(1, c["base"] + c["n"], c["kv_heads"], HEAD_DIM, dtype=torch.float16, device="cuda")
                      for _ in range(2))
        s.kv = kv_handle(s.kc, s.vc, c, 1, c["base"] + c["n"])
        s.b = {name: handle(getattr(s, name))
               for name in ("x", "w", "q", "k", "v", "gate", "up", "y", "normed", "act")}
        s.yarn = F.GhYarn(**yarn_of())
    else:
        s.logits = topk_inputs(c, seed)
        s.buf = handle(s.logits)
        s.index, s.value, s.count = np.zeros(c["k"], np.uint32), np.zeros(c["k"], np.float32), C.c_uint64()
    torch.cuda.synchronize()  # the backend has a stream of its own
    return s


# ---- one pass ----

class _Yarn:
    """The backend's rope calls take an object with c()."""

    def __init__(self, y):
        self.y = y

    def c(self):
        return self.y


def run(s):
    c, hip = s.case, backend()
    if c["kind"] == "decode":
        token = s.model.decode_greedy(int(s.tokens[0]), c["base"], 1)[0]
        logits = s.model.read_logits()
        # the chosen token's logit: the token itself may differ where two logits tie
        return {"logits": logits, "chosen": logits[token:token + 1], "k": s.k[:, c["base"]], "v": s.v[:, c["base"]]}
    if c["kind"] == "prefill":
        s.model.prefill(s.tokens, c["base"])
        rows = slice(c["base"], c["base"] + c["n"])
        return {"logits": s.model.read_logits(), "k": s.k[:, rows], "v": s.v[:, rows]}
    if c["kind"] == "topk":
        rc = hip.lib.gh_read_topk(hip.h, C.byref(s.buf), c["vocab"], c["k"], s.index.ctypes.data, s.value.ctypes.data,
                                  C.byref(s.count))
        if rc or s.count.value != min(c["k"], c["vocab"]):
            raise RuntimeError("gh_read_topk: %d" % rc)
        return {"index": s.index.astype(np.int64), "value": s.value}
    hip.begin()
    if c["kind"] == "gemm":
        x, outs = s.bufs
        for w, out in zip(s.weights, outs):
            if c["n"] == 1:
                hip.matmul(out, x, w, c["in_dim"], c["out_dim"])
            else:
                hip.matmul_batched(out, x, w, c["in_dim"], c["out_dim"], c["n"])
        result = s.out
    elif c["kind"] == "glue":
        b, n, heads = s.b, c["n"], c["kv_heads"] * c["group"]
        at = c["base"] * c["kv_heads"] * HEAD_DIM * 2
        hip.rmsnorm_x(b["normed"], b["x"], b["w"], c["d"], 1e-5, n)
        hip.rope_yarn_batched(b["q"], b["k"], heads, c["kv_heads"], HEAD_DIM, c["base"], n, _Yarn(s.yarn))
        hip.kv_write(s.kv, b["k"], b["v"], at, at, n * c["kv_heads"])
        hip.silu_mul(b["act"], b["gate"], b["up"], n * c["ffn"])
        hip.residual_add(b["x"], b["y"], n * c["d"])
        result = {"normed": s.normed, "q": s.q, "k": s.kc[0, c["base"]:], "v": s.vc[0, c["base"]:], "act": s.act,
                  "x": s.x}
    else:
        heads = c["kv_heads"] * c["group"]
        for li, (out, q) in enumerate(zip(*s.bufs)):
            if c["kind"] == "attn_decode":
                hip.attention_decode(out, q, s.kv, heads, c["base"], li)
            else:
                hip.attention_prefill(out, q, s.kv, heads, c["base"], c["n"], li)
        result = s.out
    hip.submit()
    return result


# ---- the same in 64 bits ----

def dequant(fmt, blk, rows):
    """[rows][in_dim] float64 weights of GGUF blocks."""
    nb = blk.shape[0]
    if fmt == Q4K:
        d = blk[:, :4].contiguous().view(torch.float16).double()
        sc = blk[:, 4:16].int()
        lo, hi = sc[:, :4], sc[:, 8:]
        scale = torch.cat([lo & 63, (hi & 15) | (lo >> 6 << 4)], 1).double() * d[:, :1]
        least = torch.cat([sc[:, 4:8] & 63, (hi >> 4) | (sc[:, 4:8] >> 6 << 4)], 1).double() * d[:, 1:]
        qs = blk[:, 16:].view(nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(nb, 8, 32).double()
        w = q.mul_(scale[:, :, None]).sub_(least[:, :, None])
    else:
        d = blk[:, 208:].contiguous().view(torch.float16).double()
        scale = blk[:, 192:208].contiguous().view(torch.int8).double().view(nb, 2, 4, 2, 1) * d[:, :, None, None, None]
        ql, qh = blk[:, :128].view(nb, 2, 2, 32), blk[:, 128:192].view(nb, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)  # quarters 0..3 of each half
        high = torch.cat([qh >> (2 * k) & 3 for k in range(4)], 2)
        q = (low | high << 4).double().sub_(32).view(nb, 2, 4, 2, 16)
        w = q.mul_(scale)
    return w.reshape(rows, -1)


def rms(x, w, eps=1e-5):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def silu(x):
    return x / (1 + torch.exp(-x))


def rope(x, base, query):
    """x [n][heads][128] at positions base..: adjacent pairs rotated by YaRN's angles."""
    y = yarn_of()
    pos = torch.arange(base, base + x.shape[0], device=x.device, dtype=torch.float64)
    pair = torch.arange(HEAD_DIM // 2, device=x.device, dtype=torch.float64)

    def corr(rotations):
        return y["rope_dim"] * math.log(y["original_context"] / (rotations * 2 * math.pi)) / (2 * math.log(y["freq_base"]))

    start, end = max(math.floor(corr(y["beta_fast"])), 0), min(math.ceil(corr(y["beta_slow"])), y["rope_dim"] - 1)
    keep = 1 - ((pair - start) / max(end - start, 0.001)).clamp(0, 1)
    freq = y["freq_base"] ** (-2 * pair / y["rope_dim"])
    theta = pos[:, None] * (freq / y["factor"] * (1 - keep) + freq * keep)
    cos, sin = theta.cos()[:, None], theta.sin()[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    out = torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(x.shape)
    if query:
        out = out * (1 + y["q_temperature_scale"] * torch.log((pos // y["original_context"]) + 1))[:, None, None]
    return out


def attend(q, k, v, base):
    """Causal attention of q [n][heads][128] at positions base.. over k, v [base + n][kv heads][128]."""
    n, heads = q.shape[:2]
    group = heads // k.shape[1]
    out = torch.empty_like(q)
    hidden = torch.arange(k.shape[0], device=q.device)[None] > torch.arange(base, base + n, device=q.device)[:, None]
    for h in range(heads):
        kh, vh = k[:, h // group].contiguous(), v[:, h // group].contiguous()
        s = (q[:, h].contiguous() @ kh.t().contiguous()) / math.sqrt(HEAD_DIM)
        out[:, h] = torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ vh
    return out


def exact_model(c, seed):
    n, base, heads = c["n"], c["base"], c["kv_heads"] * c["group"]
    data = model_inputs(c, seed)
    table = next(data)[3]
    out_norm, output = next(data)[3], next(data)[3]
    layers = []
    # the token ids come last: the inputs are made twice rather than all of them kept in 64 bits
    for item in model_inputs(c, seed):
        if item[1] == "tokens":
            tokens = item[3]
    per_row = c["d"] // 256
    rows = table.view(c["vocab"], per_row * BLOCK_BYTES[Q4K])[tokens].view(n * per_row, BLOCK_BYTES[Q4K])
    x = dequant(Q4K, rows, n)
    ks, vs = [], []
    for _ in range(c["blocks"]):
        an, fn = (next(data)[3].half().double() for _ in range(2))
        names = iter(LAYER)

        def project(t):
            name, _, fmt = next(names)
            return t @ dequant(fmt, next(data)[3], dims(c)[name][1]).t()

        t = rms(x, an)
        q, k, v = project(t), project(t), project(t)
        o, gate, up, down = (next(data)[3] for _ in range(4))
        old_k, old_v = (z.double() for z in next(data)[3])
        q = rope(q.view(n, heads, HEAD_DIM), base, True)
        k = rope(k.view(n, c["kv_heads"], HEAD_DIM), base, False)
        v = v.view(n, c["kv_heads"], HEAD_DIM)
        ks.append(k)
        vs.append(v)
        a = attend(q, torch.cat([old_k, k]), torch.cat([old_v, v]), base).view(n, -1)
        x = x + a @ dequant(Q4K, o, c["d"]).t()
        t = rms(x, fn)
        act = silu(t @ dequant(Q4K, gate, c["ffn"]).t()) * (t @ dequant(Q4K, up, c["ffn"]).t())
        x = x + act @ dequant(Q6K, down, c["d"]).t()
    logits = rms(x[-1], out_norm.half().double()) @ dequant(Q6K, output, c["vocab"]).t()
    k, v = torch.stack(ks), torch.stack(vs)
    if c["kind"] == "decode":
        return {"logits": logits, "chosen": logits.max().view(1), "k": k[:, 0], "v": v[:, 0]}
    return {"logits": logits, "k": k, "v": v}


def exact(case, seed):
    c = case
    if c["kind"] in ("decode", "prefill"):
        return exact_model(c, seed)
    if c["kind"] == "gemm":
        data = gemm_inputs(c, seed)
        x = next(data).double()
        return torch.stack([x @ dequant(c["fmt"], b, c["out_dim"]).t() for b in data])
    if c["kind"] == "topk":
        return {"index": None, "value": torch.topk(topk_inputs(c, seed).double(), c["k"]).values}
    if c["kind"] == "glue":
        t = {name: x.double() for name, x in glue_inputs(c, seed).items()}
        return {"normed": rms(t["x"], t["w"]), "q": rope(t["q"], c["base"], True), "k": rope(t["k"], c["base"], False),
                "v": t["v"], "act": silu(t["gate"]) * t["up"], "x": t["x"] + t["y"]}
    k, v, q = (t.double() for t in attn_inputs(c, seed))
    return torch.stack([attend(q[li], k[li], v[li], c["base"]) for li in range(c["layers"])])


def tolerance(case):
    """Four times what the present path shows against exact(): FP16 results of FP32 sums in the single
    operations (2e-4 to 3e-4), a walk of FP16 activations through the blocks in the models (1e-3 over
    eight blocks, 2e-3 over 34). RoPE, the residual sum and the appended values have no sums to reorder."""
    c = case
    if c["kind"] == "topk":
        return "exact"
    if c["kind"] in ("decode", "prefill"):
        return {"rel": 7e-3, "max": 5e-2} if c["blocks"] > 8 else {"rel": 4e-3, "max": 2.5e-2}
    return {"rel": 1.2e-3, "max": 1e-2}
