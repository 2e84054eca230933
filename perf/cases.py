"""The work that users of cwen_amd have it do, as cases that can be timed.

Seven kinds, each through the package's public entry points:

  gemv     one projection of a verify block: gemvb (all quantized formats)
  pair     the attention k and v projections of a block: gemvb_pair
  ffn      the block FFN with its residual add: mlp_block, or
           mlp_block_noalloc in programs that keep no context scratch
  head     the LM head of a block with argmax and the draft walk: head_verify
  gdn      two GatedDeltaNet verify blocks of a layer with a partial accept
           between them: GDN.block, GDN.commit
  prefill  a request's prompt through the whole model: generate_serial
  decode   serial steps and verify cycles after a long context: verify

`listed` holds the ordinary sizes; `draw` spreads sizes, block lengths and
formats over the ranges that they stand for.  Sizes are those of the 27B-shape
decoder (d 5120, FFN 17408, 24/4 heads of 256, 16/48 linear heads, vocab
151936) that the benchmark and tests use, of smaller generic decoders, and odd
ones.  `exact` is plain torch in 64 bits from the formats' definitions.
"""
import math

import torch

from cwen_amd import gpu

DEV = "cuda"
TYPES = {"q4_0": gpu.T_Q4_0, "q4_0rs": gpu.T_Q4_0RS, "q4_0rsi": gpu.T_Q4_0RSI, "q4_1": gpu.T_Q4_1,
         "q5_k": gpu.T_Q5_K, "q6_k": gpu.T_Q6_K, "q8_0": gpu.T_Q8_0}
# Reference bytes per weight of one side.
BYTES = {"q4_0": 18 / 32, "q4_0rs": 18 / 32, "q4_0rsi": 18 / 32, "q4_1": 20 / 32, "q5_k": 176 / 256,
         "q6_k": 210 / 256, "q8_0": 34 / 32}

# Decoder shapes of the whole-model cases: the 27B shape's layers, and a
# smaller one.  A model of 4 layers is one period of the hybrid pattern
# (three GatedDeltaNet layers, one full-attention layer).
SHAPES = {
    "27b": dict(n_layers=4, d_model=5120, d_ffn=17408, vocab=32768, n_head=24, n_kv_head=4, head_dim=256,
                n_rot_pairs=32, n_rot=64, gdn_nkh=16, gdn_nvh=48, gdn_dk=128, full_interval=4, max_ctx=32768,
                rope_theta=1e7, rms_eps=1e-6),
    "small": dict(n_layers=4, d_model=2048, d_ffn=6144, vocab=32000, n_head=16, n_kv_head=4, head_dim=256,
                  n_rot_pairs=32, n_rot=64, gdn_nkh=8, gdn_nvh=16, gdn_dk=128, full_interval=4, max_ctx=32768,
                  rope_theta=1e7, rms_eps=1e-6),
}


def listed():
    return [
        # the smallest calls: one token through a small, ragged projection
        {"name": "gemv_small", "kind": "gemv", "fmt": "q4_0", "M": 1000, "K": 2080, "B": 1},
        # a square projection of the 27B shape, one token
        {"name": "gemv_square", "kind": "gemv", "fmt": "q4_0", "M": 5120, "K": 5120, "B": 1},
        # the GatedDeltaNet output projection in the mixed-type files' format
        {"name": "gemv_q5k", "kind": "gemv", "fmt": "q5_k", "M": 5120, "K": 6144, "B": 8},
        # an 8-bit projection of odd sizes and a short block
        {"name": "gemv_q8_odd", "kind": "gemv", "fmt": "q8_0", "M": 3001, "K": 4128, "B": 5},
        # attention k and v of a full block
        {"name": "pair_kv", "kind": "pair", "M": 1024, "K": 5120, "B": 16},
        # the FFN: serial decode, an ordinary verify block, and a smaller
        # decoder's FFN at a full block
        {"name": "ffn_b1", "kind": "ffn", "d": 5120, "ffn": 17408, "B": 1, "noalloc": False},
        {"name": "ffn_b8", "kind": "ffn", "d": 5120, "ffn": 17408, "B": 8, "noalloc": False},
        {"name": "ffn_mid", "kind": "ffn", "d": 2048, "ffn": 5632, "B": 16, "noalloc": True},
        # the LM head of a verify block
        {"name": "head", "kind": "head", "M": 151936, "K": 5120, "B": 8, "E": 7},
        # a linear-attention layer's verify block, a partial accept, the next block
        {"name": "gdn", "kind": "gdn", "nkh": 16, "nvh": 48, "B": 8, "keep": 5},
        # a request's prompt
        {"name": "prefill", "kind": "prefill", "shape": "27b", "n": 4096},
        # serial steps and verify cycles behind that prompt
        {"name": "decode", "kind": "decode", "shape": "27b", "ctx": 4096, "B": 8, "serial": 6, "cycles": 6},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv"] * 4 + ["pair", "ffn", "ffn", "head", "gdn", "prefill", "decode"])
    B = rng.randint(1, 16)
    if kind == "gemv":
        fmt = rng.choice(["q4_0", "q4_0rs", "q4_1", "q5_k", "q6_k", "q8_0"])
        unit = 256 if fmt in ("q5_k", "q6_k") else 32
        return {"kind": kind, "fmt": fmt, "M": _log(rng, 64, 20000), "K": unit * _log(rng, max(1, 512 // unit), 17408 // unit),
                "B": B}
    if kind == "pair":
        return {"kind": kind, "M": _log(rng, 64, 4096), "K": 32 * _log(rng, 16, 256), "B": B}
    if kind == "ffn":
        return {"kind": kind, "d": 32 * _log(rng, 16, 192), "ffn": 32 * _log(rng, 32, 544), "B": B,
                "noalloc": rng.random() < 0.5}
    if kind == "head":
        return {"kind": kind, "M": _log(rng, 8000, 151936), "K": 256 * _log(rng, 4, 20), "B": B, "E": rng.randint(0, B - 1)}
    if kind == "gdn":
        nkh, nvh = rng.choice([(16, 48), (16, 32), (8, 16), (4, 4), (5, 15)])
        return {"kind": kind, "nkh": nkh, "nvh": nvh, "B": B, "keep": rng.randint(0, B)}
    shape = rng.choice(["27b", "small"])
    if kind == "prefill":
        return {"kind": kind, "shape": shape, "n": _log(rng, 8, 4096)}
    return {"kind": kind, "shape": shape, "ctx": _log(rng, 32, 8192), "B": rng.randint(2, 16), "serial": 6, "cycles": 6}


# ---------------------------------------------------------------- inputs
class _Source:
    """Seeded values on the GPU: the same for the same seed and order."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(1_000_003 * int(seed) + 17)

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device=DEV, generator=self.g)

    def normal(self, *shape):
        return torch.randn(shape, dtype=torch.float32, device=DEV, generator=self.g)

    def uniform(self, *shape):
        return torch.rand(shape, dtype=torch.float32, device=DEV, generator=self.g)

    def ints(self, n, high):
        return torch.randint(0, high, (n,), dtype=torch.int32, device=DEV, generator=self.g)

    def scale(self, sigma, n):
        """f16 |N(0, sigma)|."""
        return (self.normal(n) * sigma).abs().half()

    def weight(self, fmt, M, K):
        """A quantized matrix in its reference layout: (fmt, M, K, data bytes, f16 scales or None)."""
        if fmt in ("q5_k", "q6_k"):
            size = 176 if fmt == "q5_k" else 210
            blk = self.bytes(M * (K // 256), size)
            if fmt == "q5_k":
                blk[:, 0:2] = self.scale(0.002, blk.shape[0])[:, None].view(torch.uint8)
                blk[:, 2:4] = self.scale(0.002, blk.shape[0])[:, None].view(torch.uint8)
            else:
                blk[:, 208:210] = self.scale(0.002, blk.shape[0])[:, None].view(torch.uint8)
            return fmt, M, K, blk, None
        n = M * (K // 32)
        if fmt == "q8_0":
            blk = self.bytes(n, 34)
            blk[:, 0:2] = self.scale(0.02 / 64, n)[:, None].view(torch.uint8)
            return fmt, M, K, blk, None
        if fmt == "q4_0rs":
            return fmt, M, K, self.bytes(n, 16), self.scale(0.02 / 8, n)
        if fmt == "q4_0rsi":
            return fmt, M, K, self.bytes(2 * n, 16), self.scale(0.02 / 8, 2 * n)
        d = self.scale(0.02 / 8, n)
        if fmt == "q4_1":  # the offset near the block's minimum, as a quantiser sets it
            m = (-(8 + self.normal(n) / 2) * d.float()).half()
            return fmt, M, K, torch.cat([d[:, None].view(torch.uint8), m[:, None].view(torch.uint8), self.bytes(n, 16)], 1), None
        return fmt, M, K, torch.cat([d[:, None].view(torch.uint8), self.bytes(n, 16)], 1), None


def _host(w):
    fmt, M, K, data, sc = w
    return TYPES[fmt], data.cpu().numpy(), None if sc is None else sc.view(torch.int16).cpu().numpy(), K, M


_context = None


def _ctx():
    global _context
    if _context is None:
        _context = gpu.Context(0)
    return _context


def _inputs(case, seed):
    """Everything a case's numbers come from, on the GPU."""
    s, kind, B = _Source(seed), case["kind"], case.get("B", 1)
    if kind in ("gemv", "pair", "head"):
        fmt = {"gemv": case.get("fmt"), "pair": "q4_0rsi", "head": "q6_k"}[kind]
        d = {"w": s.weight(fmt, case["M"], case["K"]), "x": s.normal(B, case["K"])}
        if kind == "head":
            d["drafts"] = s.ints(max(1, case["E"]), case["M"])
        return d
    if kind == "ffn":
        return {"gu": s.weight("q4_0rsi", case["ffn"], case["d"]), "down": s.weight("q4_0rs", case["d"], case["ffn"]),
                "x": s.normal(B, case["d"]), "y": s.normal(B, case["d"])}
    if kind == "gdn":
        nkh, nvh = case["nkh"], case["nvh"]
        C = (2 * nkh + nvh) * 128
        d = {"S": 0.01 * s.normal(nvh, 128, 128), "hist": s.normal(C, 3), "kw": 0.3 * s.normal(C, 4),
             "wn": 1 + 0.1 * s.normal(128)}
        for i in (0, 1):
            d["blk%d" % i] = (s.normal(B, C), s.normal(B, nvh * 128), torch.log(s.uniform(B, nvh).clamp_min(1e-3)),
                              torch.sigmoid(s.normal(B, nvh)))
        return d
    return _model_inputs(case, s)


def _model_inputs(case, s):
    c = SHAPES[case["shape"]]
    H, I, V = c["d_model"], c["d_ffn"], c["vocab"]
    C, Zh, nvh = (2 * c["gdn_nkh"] + c["gdn_nvh"]) * 128, c["gdn_nvh"] * 128, c["gdn_nvh"]
    Qo, Ko = c["n_head"] * c["head_dim"], c["n_kv_head"] * c["head_dim"]
    norm = lambda n: 1 + 0.1 * s.normal(n)
    t = {"cfg": c, "embd": s.weight("q4_0rs", V, H), "out_norm": norm(H), "head": s.weight("q6_k", V, H), "layers": []}
    for l in range(c["n_layers"]):
        y = {"norm": norm(H), "post": norm(H), "gu": s.weight("q4_0rsi", I, H), "down": s.weight("q4_0rs", H, I)}
        if l % c["full_interval"] != c["full_interval"] - 1:
            y.update(qkv=s.weight("q4_0rs", C, H), z=s.weight("q4_0rs", Zh, H), alpha=s.weight("q4_0rs", nvh, H),
                     beta=s.weight("q4_0rs", nvh, H), out=s.weight("q4_0rs", H, Zh),
                     A=-torch.exp(2 * s.uniform(nvh) - 1), dt=0.5 * s.normal(nvh), conv=0.3 * s.normal(C, 4), wn=norm(128))
        else:
            y.update(q=s.weight("q4_0rs", 2 * Qo, H), kv=s.weight("q4_0rsi", Ko, H), wo=s.weight("q4_0rs", H, Qo),
                     qn=norm(c["head_dim"]), kn=norm(c["head_dim"]))
        t["layers"].append(y)
    if case["kind"] == "prefill":
        t["prompt"] = s.ints(case["n"], V)
    else:
        t["prompt"] = s.ints(case["ctx"], V)
        t["steps"] = s.ints(case["serial"], V)
        t["blocks"] = s.ints(case["cycles"] * case["B"], V).reshape(case["cycles"], case["B"])
    return t


def _model(t):
    c = t["cfg"]
    m = gpu.Model(_ctx(), **c)

    def f32(layer, tid, v):
        m.set(layer, tid, gpu.T_F32, v.reshape(-1).cpu().numpy(), None, v.numel(), 1)

    def quant(layer, tid, w):
        ty, data, sc, K, M = _host(w)
        m.set(layer, tid, ty, data, sc, K, M)

    quant(-1, gpu.TOK_EMBD, t["embd"])
    f32(-1, gpu.OUTPUT_NORM, t["out_norm"])
    quant(-1, gpu.OUTPUT, t["head"])
    for l, y in enumerate(t["layers"]):
        f32(l, gpu.ATTN_NORM, y["norm"])
        f32(l, gpu.POST_NORM, y["post"])
        quant(l, gpu.FFN_GATE_UP, y["gu"])
        quant(l, gpu.FFN_DOWN, y["down"])
        if "qkv" in y:
            for tid, k in ((gpu.ATTN_QKV, "qkv"), (gpu.ATTN_GATE, "z"), (gpu.SSM_ALPHA, "alpha"), (gpu.SSM_BETA, "beta"),
                           (gpu.SSM_OUT, "out")):
                quant(l, tid, y[k])
            for tid, k in ((gpu.SSM_A, "A"), (gpu.SSM_DT, "dt"), (gpu.SSM_CONV, "conv"), (gpu.SSM_NORM, "wn")):
                f32(l, tid, y[k])
        else:
            for tid, k in ((gpu.ATTN_Q, "q"), (gpu.ATTN_KV, "kv"), (gpu.ATTN_OUTPUT, "wo")):
                quant(l, tid, y[k])
            f32(l, gpu.ATTN_Q_NORM, y["qn"])
            f32(l, gpu.ATTN_K_NORM, y["kn"])
    return m


def prepare(case, seed):
    kind, B, d = case["kind"], case.get("B", 1), _inputs(case, seed)
    st = {"case": case, "stream": torch.cuda.current_stream().cuda_stream}

    def weight(w):
        ty, data, sc, K, M = _host(w)
        return gpu.Weight(_ctx(), ty, data, sc, K, M)

    if kind in ("prefill", "decode"):
        st["model"] = _model(d)
        st["prompt"] = d["prompt"].cpu().numpy()
        if kind == "decode":
            st["steps"] = d["steps"].cpu().numpy()
            st["blocks"] = d["blocks"].cpu().numpy()
            st["model"].generate_serial(st["prompt"], 1)
    elif kind == "ffn":
        st.update(gu=weight(d["gu"]), down=weight(d["down"]), x=d["x"], y=d["y"])
    elif kind == "gdn":
        g = gpu.GDN(_ctx(), case["nkh"], case["nvh"])
        g.set_state(d["S"].cpu().numpy(), d["hist"].cpu().numpy())
        st.update(gdn=g, kw=d["kw"], wn=d["wn"], blocks=[d["blk0"], d["blk1"]],
                  outs=[torch.empty(B, case["nvh"] * 128, device=DEV) for _ in range(2)])
    else:
        st.update(w=weight(d["w"]), x=d["x"], y=torch.empty(B, case["M"], device=DEV))
        if kind == "pair":
            st["y1"] = torch.empty(B, case["M"], device=DEV)
        if kind == "head":
            st["drafts"] = d["drafts"]
            st["res"] = torch.empty(2 + B, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    return st


def run(state):
    c, kind, stream = state["case"], state["case"]["kind"], state["stream"]
    if kind == "gemv":
        gpu.gemvb(_ctx(), state["w"], state["x"], state["y"], c["B"], stream=stream)
        return state["y"]
    if kind == "pair":
        gpu.gemvb_pair(_ctx(), state["w"], state["x"], state["y"], state["y1"], c["B"], stream=stream)
        return state["y"], state["y1"]
    if kind == "ffn":
        if c["noalloc"]:
            gpu.mlp_block_noalloc(state["gu"], state["down"], state["x"], state["y"], c["B"], stream=stream)
        else:
            gpu.mlp_block(_ctx(), state["gu"], state["down"], state["x"], state["y"], c["B"], stream=stream)
        return state["y"]
    if kind == "head":
        gpu.head_verify(_ctx(), state["w"], state["x"], c["B"], state["res"], drafts=state["drafts"], E=c["E"],
                        logits=state["y"], stream=stream)
        return state["y"], state["res"]
    if kind == "gdn":
        g = state["gdn"]
        for (qkv, z, decay, beta), out, keep in zip(state["blocks"], state["outs"], (c["keep"], c["B"])):
            g.block(qkv, z, decay, beta, state["kw"], state["wn"], out, c["B"], stream=stream)
            g.commit(keep)
        return state["outs"]
    m = state["model"]
    if kind == "prefill":
        m.generate_serial(state["prompt"], 1)
        return m.logits((c["n"] - 1) % 16 + 1)
    if m.pos + c["serial"] + c["cycles"] + c["B"] + 1 >= m.cfg.max_ctx:  # the cache is full: start over
        m.generate_serial(state["prompt"], 1)
    for t in state["steps"]:
        m.verify([t])
    for blk in state["blocks"]:  # the drafts are random ids: each cycle keeps its pending token
        m.verify(blk)
    return m.logits(c["B"])


# ---------------------------------------------------------------- what a pass cannot do without
def _trunk_weights(c):
    """Weights of the layers' matrices (elements), and of the head."""
    H, I = c["d_model"], c["d_ffn"]
    C, Zh, nvh = (2 * c["gdn_nkh"] + c["gdn_nvh"]) * 128, c["gdn_nvh"] * 128, c["gdn_nvh"]
    Qo, Ko = c["n_head"] * c["head_dim"], c["n_kv_head"] * c["head_dim"]
    full = c["n_layers"] // c["full_interval"]
    lin = c["n_layers"] - full
    return c["n_layers"] * 3 * H * I + lin * H * (C + 2 * Zh + 2 * nvh) + full * H * (3 * Qo + 2 * Ko), H * c["vocab"], full, lin


def work(case):
    kind, B = case["kind"], case.get("B", 1)
    if kind in ("gemv", "pair", "head"):
        fmt = {"gemv": case.get("fmt"), "pair": "q4_0rsi", "head": "q6_k"}[kind]
        M = case["M"] * (2 if kind == "pair" else 1)
        return {"bytes": M * case["K"] * BYTES[fmt] + 4 * B * (case["K"] + M), "flops": 2 * B * M * case["K"]}
    if kind == "ffn":
        n = 3 * case["d"] * case["ffn"]
        return {"bytes": n * 18 / 32 + 4 * B * 3 * case["d"], "flops": 2 * B * n}
    if kind == "gdn":
        nvh = case["nvh"]
        C, S = (2 * case["nkh"] + nvh) * 128, nvh * 128 * 128
        rows = 4 * B * (C + 2 * nvh * 128 + 2 * nvh)
        return {"bytes": 2 * (2 * 4 * S + rows + 4 * C * 7), "flops": 2 * B * (8 * S + 8 * C)}
    c = SHAPES[case["shape"]]
    trunk, head, full, lin = _trunk_weights(c)
    Qo, Ko = c["n_head"] * c["head_dim"], c["n_kv_head"] * c["head_dim"]
    state = lin * c["gdn_nvh"] * 128 * 128
    wbytes = trunk * 18 / 32 + head * 210 / 256
    if kind == "prefill":
        n, R = case["n"], (case["n"] - 1) % 16 + 1
        return {"bytes": wbytes + 4 * (state + full * 2 * n * Ko + R * c["vocab"]) + n * c["d_model"] * 18 / 32,
                "flops": 2 * n * trunk + 2 * R * head + full * 2 * n * n * Qo + n * 8 * state}
    steps, cycles, ctx = case["serial"], case["cycles"], case["ctx"]
    rows = steps + cycles * B
    return {"bytes": (steps + cycles) * (wbytes + 4 * (2 * state + full * 2 * ctx * Ko)) + 4 * rows * c["vocab"],
            "flops": rows * (2 * (trunk + head) + full * 4 * ctx * Qo + 8 * state)}


# ---------------------------------------------------------------- tolerances
def tolerance(case):
    """About four times what the outputs are from 64 bits."""
    if case["kind"] == "gdn":
        # 32-bit sums through the positions of two blocks: 1.8e-7 measured
        return {"rel": 2e-6, "max": 5e-5}
    if case["kind"] in ("prefill", "decode"):
        # 16-bit operands through four layers, and the state behind a context: 3.5e-4 to 5.5e-4 measured
        return {"rel": 2e-3, "max": 0.02}
    # one or two products of 16-bit operands: 0.6e-4 to 3.9e-4 measured
    return {"rel": 1.5e-3, "max": 0.01}


# ---------------------------------------------------------------- in 64 bits
def _f16(b):
    """f16 values of the byte pairs b [..., 2], in 64 bits."""
    return b.contiguous().view(torch.float16).double()


def _nibbles(q):
    """[n, 16] bytes -> [n, 32] values: the low nibbles, then the high ones."""
    return torch.cat([q & 15, q >> 4], -1).double()


def _dense(w, side=0, rows=None):
    """The matrix (or its rows [a, b)) in 64 bits."""
    fmt, M, K, data, sc = w
    a, b = rows or (0, M)
    if fmt in ("q4_0rs", "q4_0rsi"):
        k = 2 if fmt == "q4_0rsi" else 1
        q = data.reshape(M, K // 32, k, 16)[a:b, :, side]
        s = sc.reshape(M, K // 32, k)[a:b, :, side].double()
        return ((_nibbles(q) - 8) * s[..., None]).reshape(b - a, K)
    per = 256 if fmt in ("q5_k", "q6_k") else 32
    blk = data.reshape(M, K // per, -1)[a:b]
    if fmt == "q4_0":
        v = (_nibbles(blk[..., 2:]) - 8) * _f16(blk[..., 0:2])
    elif fmt == "q4_1":
        v = _nibbles(blk[..., 4:]) * _f16(blk[..., 0:2]) + _f16(blk[..., 2:4])
    elif fmt == "q8_0":
        v = blk[..., 2:].contiguous().view(torch.int8).double() * _f16(blk[..., 0:2])
    elif fmt == "q5_k":
        s6 = blk[..., 4:16]
        lo, mid, hi = s6[..., 0:4], s6[..., 4:8], s6[..., 8:12]
        scale = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1).double() * _f16(blk[..., 0:2])
        least = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], -1).double() * _f16(blk[..., 2:4])
        qh, ql = blk[..., None, 16:48], blk[..., 48:].unflatten(-1, (4, 32))
        q = torch.stack([ql & 15, ql >> 4], -2).flatten(-3, -2)  # sub-blocks 0..7
        bit = torch.arange(8, device=DEV, dtype=torch.uint8)[:, None]
        q = (q | (((qh >> bit) & 1) << 4)).double()
        v = q * scale[..., None] - least[..., None]
    else:  # q6_k
        ql, qh = blk[..., 0:128].unflatten(-1, (2, 2, 32)), blk[..., 128:192].unflatten(-1, (2, 1, 32))
        low = torch.cat([ql & 15, ql >> 4], -2)  # quarters t = 0..3 of each half
        sh = (2 * torch.arange(4, device=DEV, dtype=torch.uint8))[:, None]
        q = (low | (((qh >> sh) & 3) << 4)).double() - 32
        s = blk[..., 192:208].contiguous().view(torch.int8).double() * _f16(blk[..., 208:210])
        v = q.flatten(-3).unflatten(-1, (16, 16)) * s[..., None]
    return v.reshape(b - a, K)


def _mul(x, w, side=0):
    """x [n, K] times the matrix's transpose, in row blocks that fit."""
    M, K = w[1], w[2]
    step = max(1, (1 << 27) // K)
    return torch.cat([x @ _dense(w, side, (a, min(M, a + step))).T for a in range(0, M, step)], 1)


def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, w, eps):
    return x * w.double() / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _delta_rule(S, hist, qkv, z, decay, beta, kw, wn, nkh):
    """Outputs [T, nvh*128] of T positions; S and hist move on in place."""
    T, nvh = qkv.shape[0], z.shape[1] // 128
    seen = torch.cat([hist.T, qkv])
    x = _silu(sum(seen[j:j + T] * kw[:, j].double() for j in range(4)))
    hist.copy_(seen[T:].T)
    q, k, v = x[:, :nkh * 128], x[:, nkh * 128:2 * nkh * 128], x[:, 2 * nkh * 128:].reshape(T, nvh, 128)
    unit = lambda u: u / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6)
    of = torch.arange(nvh, device=DEV) % nkh
    q, k = (unit(u.reshape(T, nkh, 128))[:, of] for u in (q, k))
    g, out = torch.exp(decay), torch.empty(T, nvh, 128, dtype=torch.float64, device=DEV)
    for t in range(T):
        S.mul_(g[t][:, None, None])
        kt = k[t][:, :, None]
        delta = beta[t][:, None] * (v[t] - (S * kt).sum(1))
        S.add_(kt * delta[:, None, :])
        out[t] = (S * q[t][:, :, None]).sum(1)
    out /= math.sqrt(128)
    return (_rms(out, wn, 1e-6) * _silu(z.reshape(T, nvh, 128))).reshape(T, -1)


def _attend(c, y, x):
    NH, NKV, HD = c["n_head"], c["n_kv_head"], c["head_dim"]
    n = x.shape[0]
    qg = _mul(x, y["q"]).reshape(n, NH, 2, HD)
    k, v = (_mul(x, y["kv"], s).reshape(n, NKV, HD) for s in (0, 1))
    i = torch.arange(c["n_rot_pairs"], device=DEV, dtype=torch.float64)
    ang = torch.arange(n, device=DEV, dtype=torch.float64)[:, None, None] * c["rope_theta"] ** (-i / c["n_rot"])

    def rope(u):
        r, rest = u[..., :2 * len(i)], u[..., 2 * len(i):]
        a, b = r[..., 0::2], r[..., 1::2]
        return torch.cat([torch.stack([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1).flatten(-2), rest], -1)

    q, k = rope(_rms(qg[:, :, 0], y["qn"], c["rms_eps"])), rope(_rms(k, y["kn"], c["rms_eps"]))
    mask = torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1)
    out = torch.empty(n, NH, HD, dtype=torch.float64, device=DEV)
    for h in range(NH):
        kv = h // (NH // NKV)
        s = (q[:, h] @ k[:, kv].T / math.sqrt(HD)).masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, kv]
    return _mul((out * torch.sigmoid(qg[:, :, 1])).reshape(n, NH * HD), y["wo"])


def _model_logits(t, toks, last):
    """Logits of the last `last` positions of the sequence."""
    c, eps = t["cfg"], t["cfg"]["rms_eps"]
    V, H, q, sc = c["vocab"], c["d_model"], t["embd"][3], t["embd"][4]
    at = toks.long()
    x = ((_nibbles(q.reshape(V, H // 32, 16)[at]) - 8) * sc.reshape(V, H // 32)[at].double()[..., None]).reshape(-1, H)
    for y in t["layers"]:
        u = _rms(x, y["norm"], eps)
        if "qkv" in y:
            S = torch.zeros(c["gdn_nvh"], 128, 128, dtype=torch.float64, device=DEV)
            hist = torch.zeros(y["conv"].shape[0], 3, dtype=torch.float64, device=DEV)
            decay = y["A"].double() * torch.nn.functional.softplus(_mul(u, y["alpha"]) + y["dt"].double())
            x = x + _mul(_delta_rule(S, hist, _mul(u, y["qkv"]), _mul(u, y["z"]), decay, torch.sigmoid(_mul(u, y["beta"])),
                                     y["conv"], y["wn"], c["gdn_nkh"]), y["out"])
        else:
            x = x + _attend(c, y, u)
        u = _rms(x, y["post"], eps)
        x = x + _mul(_silu(_mul(u, y["gu"], 0)) * _mul(u, y["gu"], 1), y["down"])
    return _mul(_rms(x[-last:], t["out_norm"], eps), t["head"])


def exact(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    if kind == "gemv":
        return _mul(d["x"].double(), d["w"])
    if kind == "pair":
        return tuple(_mul(d["x"].double(), d["w"], s) for s in (0, 1))
    if kind == "head":
        return _mul(d["x"].double(), d["w"]), None
    if kind == "ffn":
        x = d["x"].double()
        return d["y"].double() + _mul(_silu(_mul(x, d["gu"], 0)) * _mul(x, d["gu"], 1), d["down"])
    if kind == "gdn":
        S, hist, outs = d["S"].double(), d["hist"].double(), []
        for i, keep in ((0, case["keep"]), (1, case["B"])):
            rows = [u.double() for u in d["blk%d" % i]]
            outs.append(_delta_rule(S.clone(), hist.clone(), *rows, d["kw"], d["wn"], case["nkh"]))
            if keep:
                _delta_rule(S, hist, *(u[:keep] for u in rows), d["kw"], d["wn"], case["nkh"])
        return outs
    if kind == "prefill":
        return _model_logits(d, d["prompt"], (case["n"] - 1) % 16 + 1).cpu().numpy()
    toks = torch.cat([d["prompt"], d["steps"], d["blocks"][:-1, 0], d["blocks"][-1]])
    return _model_logits(d, toks, case["B"]).cpu().numpy()
