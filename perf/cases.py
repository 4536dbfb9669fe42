"""The work whose speed is tracked, each case through the public entry points.

A case is one call (or one short sequence of calls) that a user of this library
makes: the quantizers, the decode matvec, the batched matmul in both f32 orders,
the prefill of a prompt and a chat turn (prefill, then generation). Sizes are
those of the two benchmark models (the Llama-3.2-1B shape in Q8_0 and the
Qwen3-4B shape in Q4_K_M's formats), of the Llama-3.2-3B FFN and head of the
matvec benchmark, and ragged ones between them. The model cases of one layer
block keep every width of the model, with two layers and a small vocabulary.

The entry points promise results identical to the reference's bit for bit, so
every tolerance is "exact".
"""
import math

import numpy as np
import torch

from nightrun_amd import _lib, device
from nightrun_amd.model import Model

Q8_0, Q4_K, Q6_K = _lib.Q8_0, _lib.Q4_K, _lib.Q6_K
DTYPES = {"q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
ORDERS = {"scalar": _lib.ORDER_SCALAR, "avx2": _lib.ORDER_AVX2}

# layer widths of the two benchmark models
SHAPES = {
    "llama": dict(dim=2048, n_heads=32, n_kv_heads=8, head_dim=64, ffn_dim=8192, norm_eps=1e-5, rope_theta=500000.0),
    "qwen3": dict(dim=2560, n_heads=32, n_kv_heads=8, head_dim=128, ffn_dim=9728, norm_eps=1e-6,
                  rope_theta=1000000.0, recipe=dict(rope="neox")),
}
FORMATS = {
    "llama": dict(wq=Q8_0, wk=Q8_0, wv=Q8_0, wo=Q8_0, w_gate=Q8_0, w_up=Q8_0, w_down=Q8_0, embed=Q8_0),
    "qwen3": dict(wq=Q4_K, wk=Q4_K, wv=Q6_K, wo=Q4_K, w_gate=Q4_K, w_up=Q4_K, w_down=Q6_K, embed=Q6_K),
}


def listed():
    return [
        # one decode activation row of the Qwen3-4B width, quantized before a matvec: pure latency
        dict(name="quantize_q8k_row", kind="quantize", dtype="q4_k", n=2560),
        # decode: the Llama-3.2-3B FFN matvec (the benchmark's headline)
        dict(name="matvec_q4k_ffn", kind="matvec", dtype="q4_k", order="scalar", rows=8192, cols=3072),
        # decode: the Llama-3.2-3B output head, the longest matvec of a step
        dict(name="matvec_q6k_head", kind="matvec", dtype="q6_k", order="scalar", rows=128256, cols=3072),
        # decode in the x86 host's f32 order (token identity with an AVX2 host)
        dict(name="matvec_q8_avx2", kind="matvec", dtype="q8_0", order="avx2", rows=8192, cols=2048),
        # a short prompt tail on a ragged matrix
        dict(name="matmul_q8_ragged", kind="matmul", dtype="q8_0", order="scalar", rows=1531, cols=2048, batch=13),
        # prefill: Llama-3.2-1B gate|up over a whole 512-token chunk
        dict(name="matmul_q8_ffn", kind="matmul", dtype="q8_0", order="scalar", rows="8192+8192", cols=2048,
             batch=512),
        # prefill: Qwen3-4B gate|up over a whole 512-token chunk
        dict(name="matmul_q4k_ffn", kind="matmul", dtype="q4_k", order="scalar", rows="9728+9728", cols=2560,
             batch=512),
        # prefill: Qwen3-4B down at the reference's own batch size
        dict(name="matmul_q6k_down", kind="matmul", dtype="q6_k", order="scalar", rows=2560, cols=9728, batch=64),
        # prefill in the x86 host's f32 order
        dict(name="matmul_q4k_avx2", kind="matmul", dtype="q4_k", order="avx2", rows=9728, cols=2560, batch=64),
        # a long prompt through two layers of the Llama-3.2-1B shape, room left for the answer
        dict(name="prefill_llama", kind="prefill", model="llama", layers=2, vocab=4096, ctx=4096, prompt=2000),
        # a prompt a little short of one chunk through two layers of the Qwen3-4B shape
        dict(name="prefill_qwen3", kind="prefill", model="qwen3", layers=2, vocab=4096, ctx=1024, prompt=509),
        # a whole chat turn on the whole Llama-3.2-1B shape: a 997-token prompt, 48 greedy tokens
        dict(name="chat_llama_1b", kind="chat", model="llama", layers=16, vocab=128256, ctx=2048, prompt=997,
             generate=48, sample=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["quantize", "matvec", "matvec", "matmul", "matmul", "matmul", "prefill", "prefill", "chat"])
    dtype = rng.choice(["q8_0", "q4_k", "q6_k"])
    order = rng.choice(["scalar", "scalar", "avx2"])
    qk = 32 if dtype == "q8_0" else 256
    if kind == "quantize":
        return dict(kind=kind, dtype=dtype, n=qk * _log(rng, 4, 20000))
    cols = qk * _log(rng, 1024 // qk, 10240 // qk)
    if kind == "matvec":
        return dict(kind=kind, dtype=dtype, order=order, rows=_log(rng, 500, 32768), cols=cols)
    if kind == "matmul":
        n = rng.choice([1, 1, 2, 3]) if order == "scalar" else 1
        rows = "+".join(str(_log(rng, 500, 10240)) for _ in range(n))
        return dict(kind=kind, dtype=dtype, order=order, rows=rows, cols=cols, batch=_log(rng, 2, 512))
    model = rng.choice(["llama", "qwen3"])
    prompt = _log(rng, 16, 3000)
    if kind == "prefill":
        return dict(kind=kind, model=model, layers=2, vocab=4096, ctx=prompt + rng.choice([8, 256, 1024]),
                    prompt=prompt)
    gen = rng.randint(8, 64)
    return dict(kind=kind, model=model, layers=2, vocab=4096, ctx=prompt + gen, prompt=prompt, generate=gen,
                sample=rng.random() < 0.5)


# ---- quantized tensors in the reference's block layouts, made on the GPU -------------------


def _round_away(x):
    return torch.trunc(x + torch.copysign(torch.full_like(x, 0.5), x))


def _u8(t):
    return t.contiguous().view(torch.uint8)


def _pack_q8_0(x):
    """Blocks of 32: d = amax/127 in f16, int8 quants. Returns (bytes, values)."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    d = (b.abs().amax(-1, keepdim=True) / 127).half()
    df = d.to(x.dtype)
    q = _round_away(b / torch.where(df > 0, df, torch.ones_like(df))).clamp(-127, 127)
    raw = torch.cat([_u8(d), _u8(q.to(torch.int8))], -1)
    return raw.reshape(*x.shape[:-1], -1), (q.double() * d.double()).reshape(x.shape)


def _pack_q8_k(x):
    """Activation blocks of 256: iscale = -128 / (value of largest magnitude), 16-value sums."""
    b = x.reshape(*x.shape[:-1], -1, 256)
    mx = b.gather(-1, b.abs().argmax(-1, keepdim=True))
    iscale = torch.where(mx != 0, -128.0 / mx, torch.zeros_like(mx))
    q = _round_away(b * iscale).clamp(-128, 127)
    d = torch.where(mx != 0, 1.0 / iscale, torch.zeros_like(mx)).float()
    sums = q.reshape(*q.shape[:-1], 16, 16).sum(-1)
    raw = torch.cat([_u8(d), _u8(q.to(torch.int8)), _u8(sums.to(torch.int16))], -1)
    return raw.reshape(*x.shape[:-1], -1), (q.double() * d.double()).reshape(x.shape)


def _pack_q4_k(x):
    """Blocks of 256: eight sub-blocks of 32 with 6-bit scales and mins, 4-bit quants."""
    b = x.reshape(*x.shape[:-1], -1, 8, 32)
    lo = b.amin(-1).clamp(max=0)
    scale, mn = (b.amax(-1) - lo) / 15, -lo
    d, dmin = (scale.amax(-1, keepdim=True) / 63).half(), (mn.amax(-1, keepdim=True) / 63).half()
    sc = torch.round(scale / d.to(x.dtype)).clamp(0, 63)
    m = torch.round(mn / dmin.to(x.dtype)).clamp(0, 63)
    s, o = (sc * d.to(x.dtype))[..., None], (m * dmin.to(x.dtype))[..., None]
    q = torch.round((b + o) / torch.where(s > 0, s, torch.ones_like(s))).clamp(0, 15)
    val = q.double() * (sc.double() * d.double())[..., None] - (m.double() * dmin.double())[..., None]
    si, mi, qi = sc.to(torch.uint8), m.to(torch.uint8), q.to(torch.uint8)
    head = torch.cat([si[..., :4] | (si[..., 4:] >> 4) << 6, mi[..., :4] | (mi[..., 4:] >> 4) << 6,
                      (si[..., 4:] & 15) | (mi[..., 4:] & 15) << 4], -1)
    qp = qi.reshape(*qi.shape[:-2], 4, 2, 32)
    qs = (qp[..., 0, :] | qp[..., 1, :] << 4).flatten(-2)
    raw = torch.cat([_u8(d), _u8(dmin), head, qs], -1)
    return raw.reshape(*x.shape[:-1], -1), val.reshape(x.shape)


def _pack_q6_k(x):
    """Blocks of 256: sixteen groups of 16 with int8 scales, 6-bit quants."""
    b = x.reshape(*x.shape[:-1], -1, 16, 16)
    # the value of largest magnitude maps to -32, so a group's scale has its opposite sign
    scale = b.gather(-1, b.abs().argmax(-1, keepdim=True))[..., 0] / -32
    d = (scale.gather(-1, scale.abs().argmax(-1, keepdim=True)) / -128).half()
    sc = torch.round(scale / d.to(x.dtype)).clamp(-128, 127)
    s = (sc * d.to(x.dtype))[..., None]
    q = torch.round(b / torch.where(s != 0, s, torch.ones_like(s))).clamp(-32, 31)
    val = q.double() * (sc.double() * d.double())[..., None]
    u = (q + 32).to(torch.uint8).reshape(*q.shape[:-2], 2, 4, 32)  # [half][plane][l]
    ql = torch.cat([(u[..., 0, :] & 15) | (u[..., 2, :] & 15) << 4, (u[..., 1, :] & 15) | (u[..., 3, :] & 15) << 4],
                   -1).flatten(-2)
    qh = (u[..., 0, :] >> 4 | (u[..., 1, :] >> 4) << 2 | (u[..., 2, :] >> 4) << 4 | (u[..., 3, :] >> 4) << 6).flatten(-2)
    raw = torch.cat([ql, qh, _u8(sc.to(torch.int8)), _u8(d)], -1)
    return raw.reshape(*x.shape[:-1], -1), val.reshape(x.shape)


PACK_W = {Q8_0: _pack_q8_0, Q4_K: _pack_q4_k, Q6_K: _pack_q6_k}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weights(dtype, rows, cols, g):
    """A matrix as initialized or trained ones are: normal values of std 1/sqrt(cols)."""
    x = torch.randn(rows, cols, generator=g, device="cuda") / math.sqrt(cols)
    return PACK_W[dtype](x)


def _acts(dtype, batch, cols, g):
    """Normed activations: normal, with the few large channels that language models show."""
    x = torch.randn(batch, cols, generator=g, device="cuda")
    gain = torch.where(torch.rand(cols, generator=g, device="cuda") < 0.005, 6.0, 1.0)
    return (_pack_q8_0 if dtype == Q8_0 else _pack_q8_k)(x * gain)


def _rows(case):
    """The row counts of a case's matrices: one number, or several that share the activation."""
    return [int(r) for r in str(case["rows"]).split("+")]


def _op_inputs(case, seed):
    g = _gen(seed)
    dtype = DTYPES[case["dtype"]]
    rows = _rows(case)
    ws = [_weights(dtype, r, case["cols"], g) for r in rows]
    return dtype, rows, ws, _acts(dtype, case.get("batch", 1), case["cols"], g)


# ---- models -------------------------------------------------------------------------------


def _model_weights(case, seed):
    """(weights for Model.set_weights, prompt, the 64-bit values of every tensor)."""
    c, fmt, g = SHAPES[case["model"]], FORMATS[case["model"]], _gen(seed)
    att, kv = c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    sizes = dict(wq=(att, c["dim"]), wk=(kv, c["dim"]), wv=(kv, c["dim"]), wo=(c["dim"], att),
                 w_gate=(c["ffn_dim"], c["dim"]), w_up=(c["ffn_dim"], c["dim"]), w_down=(c["dim"], c["ffn_dim"]))

    def norm(n):
        return 1.0 + 0.1 * torch.randn(n, generator=g, device="cuda")

    def tensor(name, rows, cols):
        return _weights(fmt[name], rows, cols, g)

    yield "embed", tensor("embed", case["vocab"], c["dim"])
    yield "out_norm", norm(c["dim"])
    for layer in range(case["layers"]):
        for name, (rows, cols) in sizes.items():
            yield (layer, name), tensor(name, rows, cols)
        yield (layer, "attn_norm"), norm(c["dim"])
        yield (layer, "ffn_norm"), norm(c["dim"])
        if case["model"] == "qwen3":
            yield (layer, "q_norm"), norm(c["head_dim"])
            yield (layer, "k_norm"), norm(c["head_dim"])
    yield "prompt", torch.randint(0, case["vocab"], (case["prompt"],), generator=g, device="cuda")


def _prepare_model(case, seed):
    fmt = FORMATS[case["model"]]
    w = {"embed_dtype": fmt["embed"], "layers": [{"dtypes": fmt} for _ in range(case["layers"])]}
    for key, t in _model_weights(case, seed):
        a = (t[0] if isinstance(t, tuple) else t).cpu().numpy()
        if isinstance(key, tuple):
            w["layers"][key[0]][key[1]] = a
        else:
            w[key] = a
    m = Model(dict(SHAPES[case["model"]], n_layers=case["layers"], vocab=case["vocab"]), ctx=case["ctx"])
    prompt = w.pop("prompt").astype(np.uint32)
    m.set_weights(w)
    return dict(case=case, model=m, prompt=prompt, seed=seed)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _model_logits(case, seed):
    """The prompt's last logits in 64 bits: the same path with its quantized activations and
    its f16 cache, every sum and function in 64 bits. An activation close to a rounding
    boundary quantizes to the neighbouring value here and there, and later layers carry
    that on: f32 logits lie up to a few percent from these, one layer's about 1e-7."""
    c, fmt = SHAPES[case["model"]], FORMATS[case["model"]]
    eps, hd, nh, nkv = c["norm_eps"], c["head_dim"], c["n_heads"], c["n_kv_heads"]
    tensors = dict(_model_weights(case, seed))

    def mat(key):
        return tensors[key][1]

    def lin(x, key, name):
        q = (_pack_q8_0 if fmt[name] == Q8_0 else _pack_q8_k)(x)[1]
        return q @ mat(key).t()

    prompt = tensors["prompt"]
    n = prompt.numel()
    x = mat("embed")[prompt]
    freq = (torch.tensor(c["rope_theta"], dtype=torch.float32).cuda() **
            (-2.0 * torch.arange(hd // 2, device="cuda", dtype=torch.float32) / hd))
    ang = (torch.arange(n, device="cuda", dtype=torch.float32)[:, None] * freq).double()
    cs, sn = ang.cos()[:, None], ang.sin()[:, None]

    def rope(t):  # [n][heads][hd]
        if c.get("recipe", {}).get("rope") == "neox":
            a, b = t[..., :hd // 2], t[..., hd // 2:]
            return torch.cat([a * cs - b * sn, a * sn + b * cs], -1)
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack([a * cs - b * sn, a * sn + b * cs], -1).flatten(-2)

    mask = torch.ones(n, n, device="cuda", dtype=torch.bool).tril()
    for l in range(case["layers"]):
        h = _rms(x, tensors[(l, "attn_norm")].double(), eps)
        q = lin(h, (l, "wq"), "wq").reshape(n, nh, hd)
        k = lin(h, (l, "wk"), "wk").reshape(n, nkv, hd)
        v = lin(h, (l, "wv"), "wv").reshape(n, nkv, hd)
        if case["model"] == "qwen3":
            q = _rms(q, tensors[(l, "q_norm")].double(), eps)
            k = _rms(k, tensors[(l, "k_norm")].double(), eps)
        q, k, v = rope(q), rope(k).half().double(), v.half().double()
        out = torch.empty(n, nh, hd, dtype=torch.float64, device="cuda")
        for i in range(nh):
            j = i // (nh // nkv)
            s = (q[:, i] @ k[:, j].t()) / math.sqrt(hd)
            out[:, i] = s.masked_fill(~mask, -math.inf).softmax(-1) @ v[:, j]
        x = x + lin(out.reshape(n, nh * hd), (l, "wo"), "wo")
        h = _rms(x, tensors[(l, "ffn_norm")].double(), eps)
        gate, up = lin(h, (l, "w_gate"), "w_gate"), lin(h, (l, "w_up"), "w_up")
        x = x + lin(gate * torch.sigmoid(gate) * up, (l, "w_down"), "w_down")
    return lin(_rms(x[-1:], tensors["out_norm"].double(), eps), "embed", "embed")[0]


# ---- the interface ------------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "chat"):
        return _prepare_model(case, seed)
    if kind == "quantize":
        src = torch.randn(case["n"], generator=_gen(seed), device="cuda")
        dtype = DTYPES[case["dtype"]]
        out = torch.empty(case["n"] // device.QK[dtype] * device.XBYTES[dtype], dtype=torch.uint8, device="cuda")
        return dict(case=case, src=src, out=out)
    dtype, rows, ws, (x, _) = _op_inputs(case, seed)
    ys = [torch.empty(case.get("batch", 1) * r, dtype=torch.float32, device="cuda") for r in rows]
    return dict(case=case, dtype=dtype, rows=rows, ws=[w for w, _ in ws], x=x, ys=ys)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "quantize":
        (device.quantize_q8_0 if case["dtype"] == "q8_0" else device.quantize_q8k)(state["src"], state["out"])
        return state["out"]
    if kind == "matvec":
        device.matvec(state["dtype"], ORDERS[case["order"]], state["ys"][0], state["ws"][0], state["x"],
                      case["rows"], case["cols"])
        return state["ys"]
    if kind == "matmul":
        if len(state["ws"]) > 1:
            device.matmul_group(state["dtype"], state["ys"], state["ws"], state["rows"], state["x"], case["cols"],
                                case["batch"])
        else:
            device.matmul(state["dtype"], ORDERS[case["order"]], state["ys"][0], state["ws"][0], state["x"],
                          state["rows"][0], case["cols"], case["batch"])
        return state["ys"]
    m = state["model"]
    m.reset()
    logits = m.prefill(state["prompt"])
    if kind == "prefill":
        return logits
    if case["sample"]:
        m.set_sampler(0.7, 0.9, state["seed"])
    tokens, last = m.generate(int(logits.argmax()), case["generate"], logits=True)
    return logits, tokens, last


def _model_work(case):
    c, fmt = SHAPES[case["model"]], FORMATS[case["model"]]
    att, kv = c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    sizes = dict(wq=att * c["dim"], wk=kv * c["dim"], wv=kv * c["dim"], wo=c["dim"] * att,
                 w_gate=c["ffn_dim"] * c["dim"], w_up=c["ffn_dim"] * c["dim"], w_down=c["dim"] * c["ffn_dim"])

    def stored(name, n):
        dt = fmt[name]
        return n // device.QK[dt] * device.WBYTES[dt]

    layer = sum(stored(k, n) for k, n in sizes.items())
    head = stored("embed", case["vocab"] * c["dim"])
    macs = sum(sizes.values())
    n, gen, L = case["prompt"], case.get("generate", 0), case["layers"]
    cache = 4 * kv  # f16 keys and values of one position
    byts = L * (layer + n * cache) + head + 4 * case["vocab"]
    flops = 2 * L * (n * macs + att * n * (n + 1)) + 2 * case["vocab"] * c["dim"]
    for p in range(n, n + gen):  # a decode step reads every weight and the cache so far
        byts += L * (layer + (p + 1) * cache) + head
        flops += 2 * L * (macs + 2 * att * (p + 1)) + 2 * case["vocab"] * c["dim"]
    return {"bytes": byts, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind in ("prefill", "chat"):
        return _model_work(case)
    dtype = DTYPES[case["dtype"]]
    if kind == "quantize":
        return {"bytes": 4 * case["n"] + case["n"] // device.QK[dtype] * device.XBYTES[dtype], "flops": 4 * case["n"]}
    rows = sum(_rows(case))
    batch, bpr = case.get("batch", 1), case["cols"] // device.QK[dtype]
    return {"bytes": rows * bpr * device.WBYTES[dtype] + batch * bpr * device.XBYTES[dtype] + 4 * batch * rows,
            "flops": 2 * rows * case["cols"] * batch}


def tolerance(case):
    # every entry point here is specified to the bit
    return "exact"


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None  # block bytes
    if kind in ("prefill", "chat"):
        logits = _model_logits(case, seed)
        # the generated tokens, and the logits that follow them, have no 64-bit value
        return logits if kind == "prefill" else (logits, None, None)
    _, _, ws, (_, x) = _op_inputs(case, seed)
    return [(x @ val.t()).reshape(-1) for _, val in ws]
