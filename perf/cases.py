"""The work that users of this package have it do, as timed cases.

Each case goes through the public entry points (`q8hip.*` and `Q8Llama`), over
the sizes of the model configurations in `lama32_mojo_amd/model.py`, of the
tests and of `bench.py`, plus generic and ragged sizes of the same order.  Both
packed layouts occur: groups of 64 with binary16 scales and groups of 32 with
f32 scales.  `exact` restates every case in float64 with torch alone, from the
packed bytes and the other inputs.
"""

import math

import numpy as np
import torch

from lama32_mojo_amd import model as q8model
from lama32_mojo_amd import q8hip
from lama32_mojo_amd.q8hip import Context

LAYOUTS = [(64, "f16"), (32, "f32")]
WIDTHS = [1024, 2048, 3072, 4096, 8192, 12288, 14336]
HEADS = [(32, 8, 64), (32, 8, 128), (16, 8, 128)]    # (query heads, KV heads, head_dim)
EPS = 1e-5


def listed():
    return [
        # one token's output projection of the smallest configuration: the
        # smallest call, where the launch counts
        dict(name="linear 1 row small", kind="linear", s=1, m=2048, n=1024, G=64, scale="f16"),
        # one token's norm + gate|up + swiglu of an 8B-wide block in one launch
        dict(name="fused gate-up 1 row", kind="fused", m=4096, n=28672, G=64, scale="f16"),
        # a few sequences decoded together: the long-row down projection
        dict(name="linear 4 rows", kind="linear", s=4, m=12288, n=4096, G=32, scale="f32"),
        # a batch of 16 sequences: the wide gate|up projection
        dict(name="linear 16 rows", kind="linear", s=16, m=4096, n=24576, G=32, scale="f32"),
        # a short prompt, rows and outputs at odd counts
        dict(name="linear 77 rows", kind="linear", s=77, m=4096, n=6145, G=64, scale="f16"),
        # a width whose packed rows are not 16-byte aligned
        dict(name="linear ragged width", kind="linear", s=200, m=1600, n=4800, G=64, scale="f16"),
        # a 512-row prompt with bf16 activations (the bench's prefill linears)
        dict(name="bf16 activations 512 rows", kind="bf16act", s=512, m=2048, n=16384, G=32,
             scale="f32"),
        # weights quantized and packed on the GPU when a model is prepared
        dict(name="pack", kind="pack", m=4096, n=28672, src="bf16", G=64, scale="f16"),
        # causal attention of a prompt's rows, 8B-wide heads
        dict(name="prompt attention", kind="attention", s=2048, pos0=0, nheads=32, nkv=8,
             head_dim=128),
        # one token's attention over a long cache
        dict(name="decode attention", kind="decode_attention", pos0=16000, maxlen=16384,
             nheads=32, nkv=8, head_dim=128),
        # one greedy token of a 16-layer model at 1024 cached tokens
        dict(name="decode step", kind="decode", config="Llama-3.2-1B", layers=16, pos0=1024),
        # a 2048-id prompt through 8B-wide blocks
        dict(name="prefill", kind="prefill", config="Llama-3.1-8B", layers=4, s=2048),
    ]


def log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of the listed kinds and ranges, at another size."""
    kind = rng.choice(["linear"] * 6 + ["fused", "bf16act", "bf16act", "pack", "attention",
                                        "attention", "decode_attention", "decode", "prefill"])
    G, scale = rng.choice(LAYOUTS)
    c = dict(kind=kind)
    if kind in ("linear", "bf16act"):
        c["s"] = log_int(rng, 1 if kind == "linear" else 32, 2048)
        # half the widths and output counts of the configurations, half any
        c["m"] = rng.choice(WIDTHS) if rng.random() < 0.6 else G * log_int(rng, 256 // G, 14336 // G)
        c["n"] = rng.choice(WIDTHS + [6144, 16384, 24576, 28672]) if rng.random() < 0.5 \
            else log_int(rng, 64, 32768)
        c.update(G=G, scale=scale)
    elif kind == "fused":
        c.update(m=rng.choice(WIDTHS[:5]), n=2 * log_int(rng, 512, 16384), G=G, scale=scale)
    elif kind == "pack":
        c.update(m=G * log_int(rng, 256 // G, 14336 // G), n=log_int(rng, 64, 32768),
                 src=rng.choice(["bf16", "f32"]), G=G, scale=scale)
    elif kind == "attention":
        nh, nkv, hd = rng.choice(HEADS)
        c.update(s=log_int(rng, 2, 2048), pos0=rng.choice([0, 0, log_int(rng, 1, 6000)]), nheads=nh,
                 nkv=nkv, head_dim=hd)
    elif kind == "decode_attention":
        nh, nkv, hd = rng.choice(HEADS)
        pos0 = log_int(rng, 16, 32000)
        c.update(pos0=pos0, maxlen=rng.choice([pos0 + 1, pos0 + 256, max(4096, 2 * pos0)]),
                 nheads=nh, nkv=nkv, head_dim=hd)
    elif kind == "decode":
        c.update(config=rng.choice(sorted(CONFIGS)), layers=rng.randint(2, 16),
                 pos0=log_int(rng, 16, 4000))
    else:
        c.update(config=rng.choice(sorted(CONFIGS)), layers=rng.randint(1, 4),
                 s=log_int(rng, 2, 1800))
    return c


CONFIGS = {c.name: c for c in (q8model.LLAMA_32_1B, q8model.LLAMA_31_8B, q8model.QWEN3_06B)}


def config(case):
    """The named configuration with as many of its layers as the case asks."""
    cfg = CONFIGS[case["config"]]
    return q8model.Config(**{**cfg.__dict__, "layers": min(case["layers"], cfg.layers)})


# ---- inputs -------------------------------------------------------------------

_CTX = None


def context():
    """One library context for the process, as a program keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = Context(torch.cuda.current_device())
    return _CTX


def generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def normal(shape, gen, std=1.0):
    return torch.randn(shape, device="cuda", generator=gen) * std


def rows_like_activations(s, m, gen):
    """Rows of different sizes with a few large channels, as residual
    streams and MLP activations have them."""
    x = normal((s, m), gen) * torch.exp(normal((s, 1), gen, 0.5))
    big = torch.randint(0, m, (max(1, m // 256),), device="cuda", generator=gen)
    x[:, big] *= 8.0
    return x


def wrapped(t):
    """A library view of a torch tensor, which stays alive beside it."""
    return context().wrap(t.data_ptr(), t.numel() * t.element_size())


class Packed:
    """n packed rows of m random weights in a torch tensor."""

    def __init__(self, n, m, G, scale, gen, std=0.02):
        src = normal((n, m), gen, std).to(torch.bfloat16)
        self.data = torch.empty((n, q8hip.rowstride_u16(m, G, scale)), device="cuda",
                                dtype=torch.int16)
        torch.cuda.synchronize()
        sb = wrapped(src)
        self.buf = wrapped(self.data)
        q8hip.quantize_pack(context(), sb, 0, q8hip.Q8_SRC_BF16, n, m, self.buf, 0, G, scale)
        context().sync()
        sb.free()


class Memory:
    """f32 memory of a library buffer as a torch tensor (no copy); the tensor
    keeps the buffer's owner alive."""

    def __init__(self, owner, ptr, count):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f4", "data": (ptr, False),
                                         "version": 3, "strides": None}


def prepare(case, seed):
    gen = generator(seed)
    st = globals()["prepare_" + case["kind"]](case, gen, seed)
    st["case"] = case
    torch.cuda.synchronize()
    return st


def run(state):
    return globals()["run_" + state["case"]["kind"]](state["case"], state)


def prepare_linear(c, gen, seed):
    w = Packed(c["n"], c["m"], c["G"], c["scale"], gen)
    arena = torch.empty(c["s"] * (c["m"] + c["n"]) + 4, device="cuda")
    x = arena[:c["s"] * c["m"]].view(c["s"], c["m"])
    x.copy_(rows_like_activations(c["s"], c["m"], gen))
    oy = (c["s"] * c["m"] + 3) // 4 * 4
    y = arena[oy:oy + c["s"] * c["n"]].view(c["s"], c["n"])
    return dict(w=w, arena=arena, a=wrapped(arena), x=x, oy=oy, y=y)


def run_linear(c, st):
    q8hip.linear(context(), st["w"].buf, 0, st["a"], 0, st["oy"], c["s"], c["m"], c["n"], c["G"],
                 c["scale"])
    return st["y"]


def prepare_bf16act(c, gen, seed):
    x = rows_like_activations(c["s"], c["m"], gen).to(torch.bfloat16)
    y = torch.empty((c["s"], c["n"]), device="cuda")
    return dict(w=Packed(c["n"], c["m"], c["G"], c["scale"], gen), x=x, y=y, xb=wrapped(x),
                yb=wrapped(y))


def run_bf16act(c, st):
    q8hip.linear_bf16act(context(), st["w"].buf, 0, st["xb"], 0, st["yb"], 0, c["s"], c["m"],
                         c["n"], c["G"], c["scale"])
    return st["y"]


def prepare_fused(c, gen, seed):
    m, n = c["m"], c["n"]
    rs = q8hip.rowstride_u16(m, c["G"], c["scale"])
    w = Packed(n, m, c["G"], c["scale"], gen)
    norm = (1.0 + normal((m,), gen, 0.1)).to(torch.bfloat16)
    # one weight arena: the packed rows, then the norm vector 16-byte aligned
    onorm = (n * rs + 7) // 8 * 8
    both = torch.zeros(onorm + m, device="cuda", dtype=torch.int16)
    both[:n * rs] = w.data.view(-1)
    both[onorm:] = norm.view(torch.int16)
    arena = torch.empty(m + n // 2, device="cuda")
    arena[:m] = rows_like_activations(1, m, gen)[0]
    return dict(w=w, norm=norm, both=both, wb=wrapped(both), onorm=onorm, arena=arena,
                a=wrapped(arena), x=arena[:m].view(1, m), y=arena[m:])


def run_fused(c, st):
    q8hip.linear_fused(context(), st["wb"], 0, st["a"], 0, c["m"], c["m"], c["n"], c["G"],
                       c["scale"], pre=q8hip.PRE_RMSNORM, onorm_u16=st["onorm"], eps=EPS,
                       post=q8hip.POST_SWIGLU)
    return st["y"]


def prepare_pack(c, gen, seed):
    src = normal((c["n"], c["m"]), gen, 0.02)
    if c["src"] == "bf16":
        src = src.to(torch.bfloat16)
    out = torch.empty((c["n"], q8hip.rowstride_u16(c["m"], c["G"], c["scale"])), device="cuda",
                      dtype=torch.int16)
    return dict(src=src, out=out, sb=wrapped(src), ob=wrapped(out))


def run_pack(c, st):
    code = q8hip.Q8_SRC_F32 if c["src"] == "f32" else q8hip.Q8_SRC_BF16
    q8hip.quantize_pack(context(), st["sb"], 0, code, c["n"], c["m"], st["ob"], 0, c["G"],
                        c["scale"])
    return st["out"]


def prepare_attention(c, gen, seed):
    s, hd, nh, nkv = c["s"], c["head_dim"], c["nheads"], c["nkv"]
    maxlen = c["pos0"] + s
    ldq = (nh + 2 * nkv) * hd                # q inside stacked q|k|v rows, as prompts have it
    osc = s * (ldq + nh * hd)
    arena = torch.zeros(osc + q8hip.attention_scratch_floats(s, nh, hd, maxlen) + 4, device="cuda")
    arena[:s * ldq] = normal((s * ldq,), gen)
    kv = normal((2, maxlen, nkv * hd), gen).to(torch.float16)
    return dict(arena=arena, a=wrapped(arena), kv=kv, kvb=wrapped(kv), maxlen=maxlen, ldq=ldq,
                oy=s * ldq, osc=osc, out=arena[s * ldq:osc].view(s, nh * hd))


def run_attention(c, st):
    s, hd, nh, nkv = c["s"], c["head_dim"], c["nheads"], c["nkv"]
    q8hip.attention(context(), st["a"], 0, st["kvb"], 0, st["maxlen"] * nkv * hd, st["maxlen"],
                    st["oy"], st["osc"], s, c["pos0"], nh, nkv, hd, ldq=st["ldq"])
    return st["out"]


def inv_freq(hd, theta=500000.0):
    return torch.tensor([theta ** (-2.0 * d / hd) for d in range(hd // 2)], dtype=torch.float32)


def prepare_decode_attention(c, gen, seed):
    hd, nh, nkv = c["head_dim"], c["nheads"], c["nkv"]
    qd, kvd = nh * hd, nkv * hd
    arena = torch.zeros(2 * qd + 2 * kvd + hd // 2, device="cuda")
    arena[:qd + 2 * kvd] = normal((qd + 2 * kvd,), gen)
    oinv = 2 * qd + 2 * kvd
    arena[oinv:] = inv_freq(hd).cuda()
    kv = normal((2, c["maxlen"], kvd), gen).to(torch.float16)
    return dict(arena=arena, a=wrapped(arena), kv=kv, kvb=wrapped(kv), oinv=oinv,
                oy=qd + 2 * kvd, out=arena[qd + 2 * kvd:oinv], new=kv[:, c["pos0"]])


def run_decode_attention(c, st):
    hd, nh, nkv = c["head_dim"], c["nheads"], c["nkv"]
    qd, kvd = nh * hd, nkv * hd
    q8hip.decode_attention(context(), st["a"], 0, qd, qd + kvd, st["oinv"], st["kvb"], 0,
                           c["maxlen"] * kvd, c["maxlen"], st["oy"], c["pos0"], nh, nkv, hd)
    return {"out": st["out"], "new_kv": st["new"]}


class Model:
    """A Q8Llama with random weights, and its logits as a torch tensor."""

    def __init__(self, case, seed, maxlen, rows):
        self.cfg = config(case)
        self.m = q8model.Q8Llama(context(), self.cfg, maxlen, seed=seed, max_prefill=rows)

    def __del__(self):
        self.m.close()


def prepare_decode(c, gen, seed):
    M = Model(c, seed, c["pos0"] + 16, 1)
    m, cfg = M.m, M.cfg
    kv = normal((2 * cfg.layers, m.maxlen, cfg.kv_dim()), gen).to(torch.float16).cpu()
    m.kv.upload(kv.numpy())
    m.capture_decode()
    token = int(torch.randint(0, cfg.vocab, (1,), device="cuda", generator=gen))
    logits = torch.as_tensor(Memory(M, m.a.buf.ptr + 4 * m.graph_logits, cfg.vocab),
                             device="cuda")
    return dict(model=M, kv=kv, token=token, logits=logits)


def run_decode(c, st):
    m = st["model"].m
    m.n_cached = c["pos0"]
    ids = m.decode_steps(st["token"], 1)
    return {"logits": st["logits"], "ids": ids}


def prepare_prefill(c, gen, seed):
    M = Model(c, seed, c["s"] + 16, c["s"])
    ids = torch.randint(0, M.cfg.vocab, (c["s"],), device="cuda", generator=gen).tolist()
    return dict(model=M, ids=ids)


def run_prefill(c, st):
    m = st["model"].m
    m.reset()
    return m.forward(st["ids"])


# ---- work ------------------------------------------------------------------------

def packed_bytes(n, m, G, scale):
    return n * (m + m // G * (2 if scale == "f16" else 4))


def model_linear(cfg):
    """(n, m) of a block's matrices."""
    H, QD, KVD, I = cfg.hidden, cfg.q_dim(), cfg.kv_dim(), cfg.inter
    return [(QD + 2 * KVD, H), (H, QD), (2 * I, H), (H, I)]


def work(case):
    k = case["kind"]
    if k in ("linear", "bf16act", "fused"):
        s, m, n = case.get("s", 1), case["m"], case["n"]
        xb = 2 if k == "bf16act" else 4
        out = n // 2 if k == "fused" else n
        return {"bytes": packed_bytes(n, m, case["G"], case["scale"]) + s * (xb * m + 4 * out),
                "flops": 2 * s * m * n}
    if k == "pack":
        n, m = case["n"], case["m"]
        return {"bytes": n * m * (2 if case["src"] == "bf16" else 4)
                + packed_bytes(n, m, case["G"], case["scale"]), "flops": 2 * n * m}
    if k in ("attention", "decode_attention"):
        s, p, hd = case.get("s", 1), case["pos0"], case["head_dim"]
        pairs = sum(p + i + 1 for i in range(s))
        return {"bytes": 2 * 2 * (p + s) * case["nkv"] * hd + 2 * 4 * s * case["nheads"] * hd,
                "flops": 4 * pairs * case["nheads"] * hd}
    cfg = config(case)
    s = case.get("s", 1)
    p = case.get("pos0", 0)
    mats = model_linear(cfg)
    weights = cfg.layers * sum(packed_bytes(n, m, 64, "f16") for n, m in mats) \
        + packed_bytes(cfg.vocab, cfg.hidden, 64, "f16")
    pairs = sum(p + i + 1 for i in range(s))
    return {"bytes": weights + cfg.layers * 2 * 2 * (p + s) * cfg.kv_dim() + 4 * cfg.vocab,
            "flops": cfg.layers * (2 * s * sum(n * m for n, m in mats)
                                   + 4 * pairs * cfg.q_dim()) + 2 * cfg.vocab * cfg.hidden}


def tolerance(case):
    """Four times what the paths differ by from float64: f32 arithmetic up to
    31 rows (x split into two bf16 terms from 5 on); binary16 activations and
    weights in the GEMM from 32 rows; f32 rotation angles (up to 16000 rad)
    and binary16 cache rows in the token steps; packed bytes exactly."""
    k = case["kind"]
    if k == "pack":
        return "exact"
    if k == "bf16act" or (k == "linear" and case["s"] >= 32):
        return {"rel": 1.2e-3}
    if k == "prefill":
        return {"rel": 8e-3}
    if k == "decode_attention":
        return {"rel": 8e-4}
    if k == "decode":
        return {"rel": 1e-4}
    return {"rel": 1e-5}


# ---- float64 -------------------------------------------------------------------------

def unpack(data, m, G, scale):
    """Packed rows (int16 [n, stride]) as float64 weights [n, m]."""
    n = data.shape[0]
    b = data.contiguous().view(torch.uint8).view(n, -1)
    sb = m // G * (2 if scale == "f16" else 4)
    kind = torch.float16 if scale == "f16" else torch.float32
    sc = b[:, :sb].contiguous().view(kind).to(torch.float64)
    q = b[:, sb:sb + m].contiguous().view(torch.int8).to(torch.float64)
    return (q.view(n, m // G, G) * sc[:, :, None]).view(n, m)


def rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def rotate(x, inv, pos0):
    """rotate_half RoPE of x [s, heads, hd] at positions pos0 .."""
    pos = torch.arange(pos0, pos0 + x.shape[0], device=x.device, dtype=torch.float64)
    ang = pos[:, None] * inv.to(torch.float64).to(x.device)[None]
    cs, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x.chunk(2, -1)
    return torch.cat([a * cs - b * sn, b * cs + a * sn], -1)


def attend(q, k, v, pos0):
    """Causal attention in float64: q [s, nh, hd], k and v [ctx, nkv, hd]."""
    s, nh, hd = q.shape
    grp = nh // k.shape[1]
    mask = torch.arange(k.shape[0], device=q.device)[None] > \
        (pos0 + torch.arange(s, device=q.device))[:, None]
    out = torch.empty_like(q)
    for h in range(nh):
        sc = q[:, h] @ k[:, h // grp].T / math.sqrt(hd)
        out[:, h] = torch.softmax(sc.masked_fill(mask, -math.inf), -1) @ v[:, h // grp]
    return out


def exact(case, seed):
    st = prepare(case, seed)
    k = case["kind"]
    if k == "pack":
        return None
    if k in ("linear", "bf16act"):
        w = unpack(st["w"].data, case["m"], case["G"], case["scale"])
        return st["x"].to(torch.float64) @ w.T
    if k == "fused":
        w = unpack(st["w"].data, case["m"], case["G"], case["scale"])
        g, u = (rms(st["x"].to(torch.float64), st["norm"].to(torch.float64)) @ w.T)[0].chunk(2)
        return torch.nn.functional.silu(g) * u
    if k == "attention":
        s, hd, nh = case["s"], case["head_dim"], case["nheads"]
        q = st["arena"][:s * st["ldq"]].view(s, st["ldq"])[:, :nh * hd].to(torch.float64)
        kc, vc = st["kv"].to(torch.float64).view(2, st["maxlen"], case["nkv"], hd)
        return attend(q.reshape(s, nh, hd), kc, vc, case["pos0"]).view(s, nh * hd)
    if k == "decode_attention":
        hd, nh, nkv, p = case["head_dim"], case["nheads"], case["nkv"], case["pos0"]
        a = st["arena"].to(torch.float64)
        qd, kvd = nh * hd, nkv * hd
        inv = st["arena"][st["oinv"]:]
        q = rotate(a[:qd].view(1, nh, hd), inv, p)
        kn = rotate(a[qd:qd + kvd].view(1, nkv, hd), inv, p)
        vn = a[qd + kvd:qd + 2 * kvd].view(1, nkv, hd)
        kc, vc = st["kv"].to(torch.float64).view(2, case["maxlen"], nkv, hd)[:, :p]
        out = attend(q, torch.cat([kc, kn]), torch.cat([vc, vn]), p)
        return {"out": out.view(-1), "new_kv": torch.stack([kn.view(-1), vn.view(-1)])}
    return exact_model(case, st)


def exact_model(case, st):
    M = st["model"]
    m, cfg = M.m, M.cfg
    arena = torch.from_numpy(m.w.buf.download((m.w.top,), np.int16)).cuda()
    shapes = q8model.tensor_shapes(cfg)

    def matrix(name):
        n, mm = shapes[name]
        rs = q8hip.rowstride_u16(mm, 64, "f16")
        o = m.w.o(name)
        return arena[o:o + n * rs].view(n, rs), mm

    def lin(x, name):
        data, mm = matrix(name)
        return torch.cat([x @ unpack(d, mm, 64, "f16").T for d in data.split(16384)], -1)

    def vector(name):
        o = m.w.o(name)
        return arena[o:o + shapes[name][0]].view(torch.bfloat16).to(torch.float64)

    def norm(x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + cfg.eps) * vector(name)

    p = case.get("pos0", 0)
    ids = [st["token"]] if case["kind"] == "decode" else st["ids"]
    s, hd = len(ids), cfg.head_dim
    inv = torch.from_numpy(q8model.rope_inv_freq(cfg))
    data, mm = matrix("model.embed_tokens.weight")
    h = unpack(data[torch.tensor(ids, device="cuda")], mm, 64, "f16")
    for L in range(cfg.layers):
        pre = f"model.layers.{L}."
        x = norm(h, pre + "input_layernorm.weight")
        q = lin(x, pre + "self_attn.q_proj.weight").view(s, cfg.n_heads, hd)
        k = lin(x, pre + "self_attn.k_proj.weight").view(s, cfg.n_kv, hd)
        v = lin(x, pre + "self_attn.v_proj.weight").view(s, cfg.n_kv, hd)
        if cfg.qk_norm:
            q = norm(q, pre + "self_attn.q_norm.weight")
            k = norm(k, pre + "self_attn.k_norm.weight")
        q, k = rotate(q, inv, p), rotate(k, inv, p)
        if p:
            old = st["kv"][2 * L:2 * L + 2, :p].cuda().to(torch.float64).view(2, p, cfg.n_kv, hd)
            k, v = torch.cat([old[0], k]), torch.cat([old[1], v])
        h = h + lin(attend(q, k, v, p).view(s, -1), pre + "self_attn.o_proj.weight")
        x = norm(h, pre + "post_attention_layernorm.weight")
        x = torch.nn.functional.silu(lin(x, pre + "mlp.gate_proj.weight")) \
            * lin(x, pre + "mlp.up_proj.weight")
        h = h + lin(x, pre + "mlp.down_proj.weight")
    head = "model.embed_tokens.weight" if cfg.tied else "lm_head.weight"
    logits = lin(norm(h[-1:], "model.norm.weight"), head)[0]
    if case["kind"] == "prefill":
        return logits
    return {"logits": logits, "ids": [None]}
