"""The work that a user of this framework has it do, as cases that can be timed.

Each case goes through a public entry point (tinygiant_amd.moe.MoEBlock,
tinygiant_amd.sample.Sampler, or a C-ABI symbol of include/tinygiant.h bound
by tinygiant_amd._lib), with the shapes of bench.py and the tests: the 30B
shape (embedding 2048, expert width 768, 128 experts, 8 per token), the 235B
shape (4096, 1536, 128, 8), a vocabulary of 151936.

kind "stack"   MoEBlock.step: one token (or a few) through a stack of layers,
               the decode step of an engine
kind "layer"   MoEBlock.forward: one MoE layer for a batch of tokens, from a
               few concurrent users over batched decode to prompt processing
kind "head"    tg_head_forward: output norm, fp32 vocabulary product, greedy
               token; the logits come back to the host as the engine reads them
kind "sample"  Sampler: temperature / top-p draws from logits on the device
kind "moe"     tg_moe_forward: the reference's own call, Q4_K experts in locked
               (mirrored) read-only mappings, one call per layer
kind "block"   tg_transformer_layer: the reference's whole layer, f32 attention
               over a filled KV cache and Q4_K experts, weights locked
"""
import ctypes
import math
import mmap
import tempfile

import numpy as np
import torch

from tinygiant_amd import _lib
from tinygiant_amd.arena import HBMExpertArena
from tinygiant_amd.moe import MoEBlock
from tinygiant_amd.sample import Sampler

EPS = 1e-6
SHAPES = {"30b": (2048, 768, 128, 8), "235b": (4096, 1536, 128, 8)}


def listed():
    return [
        # one user decoding: a token through all 48 layers of the 30B shape (bench.py's headline)
        {"name": "decode_stack_30b", "kind": "stack", "shape": "30b", "layers": 48, "tokens": 1, "skew": False},
        # the same for the large model, on the share of its 94 layers that is quick to fill (10.9 GB, far over the caches)
        {"name": "decode_stack_235b", "kind": "stack", "shape": "235b", "layers": 8, "tokens": 1, "skew": False},
        # a handful of concurrent users: an odd, small batch through one layer
        {"name": "layer_5_tokens", "kind": "layer", "shape": "30b", "tokens": 5, "skew": True},
        # batched decode, 64 sequences, popularity-skewed routing (bench.py's batched leg)
        {"name": "layer_64_tokens", "kind": "layer", "shape": "30b", "tokens": 64, "skew": True},
        # batched decode of the large model, 32 sequences (bench.py's 235B batched leg)
        {"name": "layer_32_tokens_235b", "kind": "layer", "shape": "235b", "tokens": 32, "skew": True},
        # a short prompt: a ragged number of tokens that fills no tile
        {"name": "layer_333_tokens", "kind": "layer", "shape": "30b", "tokens": 333, "skew": False},
        # a long prompt: bench.py's prefill leg, one layer of it
        {"name": "layer_2048_tokens", "kind": "layer", "shape": "30b", "tokens": 2048, "skew": False},
        # the step after the layers: 151936 x 2048 fp32 logits and the greedy token
        {"name": "output_head", "kind": "head", "vocab": 151936, "embed": 2048},
        # the next token of 4 sequences at the reference's defaults (temperature 0.7, top-p 0.9)
        {"name": "sample_nucleus", "kind": "sample", "vocab": 151936, "rows": 4, "temperature": 0.7, "top_p": 0.9},
        # plain temperature sampling, nothing cut off (top-p 1)
        {"name": "sample_full", "kind": "sample", "vocab": 151936, "rows": 4, "temperature": 1.0, "top_p": 1.0},
        # the reference engine's expert call on its own Q4_K experts, four layers' calls one after another
        {"name": "q4k_moe", "kind": "moe", "shape": "30b", "calls": 4, "experts": 8},
        # the reference's whole decode layer at 1024 cached positions
        {"name": "q4k_block", "kind": "block", "shape": "30b", "experts": 8, "heads": 32, "kv_heads": 4, "head_dim": 128,
         "kv_len": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "stack", "stack", "head", "sample", "sample", "moe", "block"])
    if kind == "layer":
        if rng.random() < 0.7:
            return {"kind": "layer", "shape": "30b", "tokens": _log_int(rng, 1, 2040), "skew": rng.random() < 0.5}
        return {"kind": "layer", "shape": "235b", "tokens": _log_int(rng, 1, 500), "skew": rng.random() < 0.5}
    if kind == "stack":
        if rng.random() < 0.6:
            return {"kind": "stack", "shape": "30b", "layers": rng.randint(6, 44), "tokens": rng.choice([1, 1, 1, 2, 3]), "skew": False}
        return {"kind": "stack", "shape": "235b", "layers": rng.randint(2, 7), "tokens": rng.choice([1, 1, 2]), "skew": False}
    if kind == "head":
        return {"kind": "head", "vocab": _log_int(rng, 32000, 151000), "embed": rng.choice([1024, 2048, 2560])}
    if kind == "sample":
        return {"kind": "sample", "vocab": _log_int(rng, 32000, 151000), "rows": rng.randint(1, 4),
                "temperature": round(rng.uniform(0.6, 1.2), 3), "top_p": rng.choice([1.0, round(rng.uniform(0.8, 0.99), 3)])}
    if kind == "moe":
        return {"kind": "moe", "shape": rng.choice(["30b", "235b"]), "calls": rng.randint(1, 4), "experts": rng.randint(4, 10)}
    return {"kind": "block", "shape": "30b", "experts": rng.randint(4, 8), "heads": rng.choice([16, 32]), "kv_heads": rng.choice([4, 8]),
            "head_dim": rng.choice([64, 128]), "kv_len": _log_int(rng, 64, 2000)}


# ------------------------------------------------------------------ inputs
def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + what * 7919 + 17) & 0x7FFFFFFFFFFF)
    return g


def _randn(seed, what, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=_gen(seed, what), device="cuda", dtype=torch.float32) * std + mean


def _q4_0(w):
    """[.., 32 n] floats -> (q [.., n, 32] uint8, d [.., n] half): the Q4_0 rule, d = m / -8 with m the signed value of
    largest magnitude."""
    b = w.reshape(*w.shape[:-1], -1, 32)
    m = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True))
    d = m / -8.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    q = torch.clamp(torch.floor(b * inv + 8.5), 0, 15).to(torch.uint8)
    return q, d.squeeze(-1).half()


def _pool_expert(seed, shape, e):
    """Expert e of the seed's pool: gate, up [I, H] and down [H, I], N(0, 0.02) in Q4_0, as (q, d) each."""
    H, I, _, _ = SHAPES[shape]
    return [_q4_0(_randn(seed, 1000 + 4 * e + t, r, c, std=0.02)) for t, (r, c) in enumerate([(I, H), (I, H), (H, I)])]


def _pool_bytes(seed, shape, n):
    """The pool's n experts as relayout bytes (gate | up | down, 18-byte blocks), in host memory."""
    H, I, _, _ = SHAPES[shape]
    out = torch.empty(n, 3 * H * I // 32 * 18, dtype=torch.uint8, device="cuda")
    for e in range(n):
        parts = []
        for q, d in _pool_expert(seed, shape, e):
            parts.append(torch.cat([d.unsqueeze(-1).contiguous().view(torch.uint8), q[..., :16] | (q[..., 16:] << 4)], -1).reshape(-1))
        out[e] = torch.cat(parts)
    return out.cpu().numpy().reshape(-1)


def _router(seed, shape, layer, skew):
    """(router [E, H], shift [H]): N(0, 0.02), and with skew a per-expert offset along a direction that every token
    shares, so that expert popularity follows a power law with exponent of about 1.1."""
    H, _, E, _ = SHAPES[shape]
    r = _randn(seed, 100 + layer, E, H, std=0.02)
    if not skew:
        return r, torch.zeros(H, device="cuda")
    u = _randn(seed, 90, H)
    u = u / u.norm()
    c = 0.5 * math.sqrt(H)
    rms = math.sqrt(1.25)  # of a token with the shift
    bias = -0.6 * (0.02 * math.sqrt(H) / rms) * torch.log(torch.arange(1, E + 1, device="cuda", dtype=torch.float32))
    return r + bias[:, None] * (rms / c) * u[None, :], c * u


def _norm(seed, shape, layer):
    return _randn(seed, 200 + layer, SHAPES[shape][0], std=0.1, mean=1.0)


def _tokens(case, seed):
    H = SHAPES[case["shape"]][0]
    return _randn(seed, 1, case["tokens"], H) + _router(seed, case["shape"], 0, case["skew"])[1]


def _q4k(seed, what, blocks):
    """Random Q4_K blocks (144 bytes each): half d and dmin, packed 6-bit scales and mins, nibbles."""
    b = torch.randint(0, 256, (blocks, 144), generator=_gen(seed, what), device="cuda", dtype=torch.uint8)
    u = torch.rand(blocks, 2, generator=_gen(seed, what + 1), device="cuda")
    dm = torch.stack([0.0005 + 0.0035 * u[:, 0], 0.004 * u[:, 1]], 1).half()
    b[:, :4] = dm.view(torch.uint8)
    return b


def _q4k_expert(seed, shape, e):
    H, I, _, _ = SHAPES[shape]
    return _q4k(seed, 5000 + 10 * e, 3 * I * H // 256)


def _expert_weights(n):
    w = np.linspace(1.0, 0.7, n)
    return (w / w.sum()).astype(np.float32)


def _readonly(parts):
    """The byte arrays in one temporary file, mapped back read-only: how the reference's cache holds its experts."""
    with tempfile.TemporaryFile() as f:
        for p in parts:
            f.write(p.tobytes())
        f.flush()
        mm = mmap.mmap(f.fileno(), 0, access=mmap.ACCESS_READ)
    views, off = [], 0
    for p in parts:
        views.append(np.frombuffer(mm, np.uint8, count=p.nbytes, offset=off))
        off += p.nbytes
    return views


class _Kept:
    """What a program keeps between calls; gives back its device copies when it goes."""

    def __init__(self, **kw):
        self.__dict__.update(kw)
        self.drop = []

    def __del__(self):
        try:
            lib = _lib.require_lib()
            for a in self.drop:
                lib.tg_mirror_drop(ctypes.c_void_p(a.ctypes.data), ctypes.c_size_t(a.nbytes))
            if getattr(self, "head", None):
                lib.tg_head_destroy(self.head)
            if getattr(self, "sampler", None):
                self.sampler.close()
            if getattr(self, "arena", None):
                self.arena.close()
        except Exception:
            pass

    def lock(self, arrays):
        lib = _lib.require_lib()
        for a in arrays:
            lib.tg_mlock(ctypes.c_void_p(a.ctypes.data), ctypes.c_size_t(a.nbytes))
            self.drop.append(a)


def _block_inputs(case, seed):
    """(attention weights q, k, v, o; norm weights attn, ffn, q, k; rope cos, sin; caches k, v; x), float32 tensors."""
    H = SHAPES[case["shape"]][0]
    hd, kvmax = case["head_dim"], 2048
    qd, kd = case["heads"] * hd, case["kv_heads"] * hd
    w = [_randn(seed, 300 + i, r, c, std=0.02) for i, (r, c) in enumerate([(qd, H), (kd, H), (kd, H), (H, qd)])]
    n = [_randn(seed, 310 + i, m, std=0.1, mean=1.0) for i, m in enumerate([H, H, hd, hd])]
    ang = np.arange(kvmax)[:, None] * (10000.0 ** (-np.arange(hd // 2) / (hd // 2)))[None, :]
    rope = [torch.from_numpy(f(ang).astype(np.float32)).cuda() for f in (np.cos, np.sin)]
    kv = [_randn(seed, 320 + i, case["kv_heads"], kvmax, hd) for i in range(2)]
    return w, n, rope, kv, _randn(seed, 330, H)


def prepare(case, seed):
    _lib.call("tg_gpu_init", 0)
    kind = case["kind"]
    if kind in ("stack", "layer"):
        H, I, E, k = SHAPES[case["shape"]]
        L = case.get("layers", 1)
        # layer l's expert e is expert l + e of a pool: every layer holds other experts in other places
        pool = _pool_bytes(seed, case["shape"], E + L - 1)
        eb = pool.nbytes // (E + L - 1)
        a = HBMExpertArena(L, E, H, I, k)
        for l in range(L):
            a.load_layer(l, pool[l * eb:(l + E) * eb])
            a.load_router(l, _router(seed, case["shape"], l, case["skew"])[0].cpu().numpy())
            a.load_norm(l, _norm(seed, case["shape"], l).cpu().numpy())
        x = _tokens(case, seed)
        torch.cuda.synchronize()
        return _Kept(kind=kind, arena=a, block=MoEBlock(a, EPS), x=x)
    if kind == "head":
        W = _randn(seed, 1, case["vocab"], case["embed"], std=0.02).cpu().numpy()
        nw = _randn(seed, 2, case["embed"], std=0.1, mean=1.0).cpu().numpy()
        h = _lib.require_lib().tg_head_create(W.ctypes.data, nw.ctypes.data, case["vocab"], case["embed"])
        if not h:
            raise RuntimeError("tg_head_create failed")
        return _Kept(kind=kind, head=h, x=_randn(seed, 3, case["embed"]).cpu().numpy(),
                     logits=np.empty(case["vocab"], np.float32))
    if kind == "sample":
        return _Kept(kind=kind, sampler=Sampler(case["vocab"]), temperature=case["temperature"], top_p=case["top_p"],
                     logits=[_randn(seed, 1 + r, case["vocab"], std=2.5) for r in range(case["rows"])],
                     u=np.random.RandomState(int(seed) & 0x7FFFFFFF).random_sample(case["rows"]))
    H, I, _, _ = SHAPES[case["shape"]]
    n, gb = case["experts"], I * H // 256 * 144
    calls = case.get("calls", 1)
    views = _readonly([_q4k_expert(seed, case["shape"], e).cpu().numpy().reshape(-1) for e in range(n * calls)])
    st = _Kept(kind=kind, H=H, I=I, n=n, views=views, w=_expert_weights(n))
    if kind == "moe":
        st.ptrs = [(ctypes.c_void_p * n)(*[v.ctypes.data for v in views[c * n:(c + 1) * n]]) for c in range(calls)]
        st.x = [_randn(seed, 400 + c, H).cpu().numpy() for c in range(calls)]
        st.lock(views)
        return st
    w, nrm, rope, kv, x = ([t.cpu().numpy() for t in v] if isinstance(v, list) else v.cpu().numpy() for v in _block_inputs(case, seed))
    st.case, st.attn, st.norms, st.rope, st.kv, st.x = case, w, nrm, rope, kv, x
    st.gp, st.up, st.dp = [(ctypes.c_void_p * n)(*[v.ctypes.data + t * gb for v in views]) for t in range(3)]
    st.fmt = np.zeros(n, np.int32)
    # the engine locks its attention weights (writable arrays, never written afterwards) and its experts
    _lib.require_lib().tg_mirror_mode(2)
    st.lock(w + nrm + views)
    return st


def run(st):
    if st.kind == "layer":
        out, idx, w = st.block.forward(0, st.x, return_routing=True)
        return {"out": out, "idx": idx, "w": w}
    if st.kind == "stack":
        return st.block.step(st.x.clone())
    if st.kind == "head":
        tok = ctypes.c_int32()
        _lib.call("tg_head_forward", st.head, st.x.ctypes.data, EPS, st.logits.ctypes.data, ctypes.byref(tok))
        return {"logits": st.logits, "token": tok.value}
    if st.kind == "sample":
        return [st.sampler(l, st.temperature, st.top_p, u=float(u)) for l, u in zip(st.logits, st.u)]
    lib = _lib.require_lib()
    if st.kind == "moe":
        outs = []
        for ptrs, x in zip(st.ptrs, st.x):
            out = np.empty(st.H, np.float32)
            lib.tg_moe_forward(ptrs, st.w.ctypes.data, st.n, x.ctypes.data, out.ctypes.data, st.H, st.I)
            outs.append(out)
        return outs
    x, c = st.x.copy(), st.case
    lib.tg_transformer_layer(*(a.ctypes.data for a in st.attn), st.norms[0].ctypes.data, st.norms[2].ctypes.data,
                             st.norms[3].ctypes.data, st.norms[1].ctypes.data, st.kv[0].ctypes.data, st.kv[1].ctypes.data,
                             c["kv_len"], 2048, st.rope[0].ctypes.data, st.rope[1].ctypes.data, st.gp, st.up, st.dp,
                             st.fmt.ctypes.data, st.w.ctypes.data, st.n, x.ctypes.data, st.H, st.I, c["heads"],
                             c["kv_heads"], c["head_dim"], c["kv_len"])
    return {"x": x, "k": st.kv[0], "v": st.kv[1]}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind in ("stack", "layer"):
        H, I, E, k = SHAPES[case["shape"]]
        T, L = case["tokens"], case.get("layers", 1)
        p = np.arange(1, E + 1) ** (-1.1 if case["skew"] else 0.0)
        p = np.minimum(1.0, k * p / p.sum())
        distinct = min(E, T * k, float(np.sum(1 - (1 - p) ** T)))
        eb = 3 * H * I // 32 * 18
        return {"bytes": L * (distinct * eb + 4 * E * H + 8 * T * H), "flops": L * 2 * T * (k * 3 * H * I + E * H)}
    if kind == "head":
        return {"bytes": 4 * (case["vocab"] * case["embed"] + case["embed"] + case["vocab"]),
                "flops": 2 * case["vocab"] * case["embed"]}
    if kind == "sample":
        return {"bytes": case["rows"] * 4 * case["vocab"], "flops": case["rows"] * 8 * case["vocab"]}
    H, I, _, _ = SHAPES[case["shape"]]
    n, calls = case["experts"], case.get("calls", 1)
    b, f = calls * (n * 3 * H * I // 256 * 144 + 8 * H), calls * 2 * n * 3 * H * I
    if kind == "block":
        qd, kd, s = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["kv_len"] + 1
        b += 4 * (2 * H * qd + 2 * H * kd) + 2 * 4 * kd * s
        f += 2 * (2 * H * qd + 2 * H * kd) + 4 * qd * s
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times what the path differs from exact() by."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "head":
        return {"rel": 1.5e-6}
    if kind == "moe":
        return {"rel": 1e-5}
    if kind == "block":  # an 8-bit value of the expert input may round the other way
        return {"rel": 1e-4}
    # an 8-bit activation, or its 16-bit scale, may round the other way, and a token's last expert may change places
    # with the next on a near tie; in a stack that travels on through the layers (8e-3 seen)
    return {"rel": 0.03} if kind == "stack" else {"rel": 2e-3, "differ": 1e-3}


# ------------------------------------------------------------------ the same in 64 bits, in plain torch
def _q8(v, group, half_scale):
    """v through its 8-bit form per group: values q = rint(127 v / amax), scale amax / 127 (as a half)."""
    b = v.reshape(*v.shape[:-1], -1, group)
    a = b.abs().amax(-1, keepdim=True)
    q = torch.where(a > 0, torch.round(b * (127.0 / torch.clamp(a, min=1e-300))), torch.zeros_like(b))
    d = a / 127.0
    if half_scale:
        d = d.float().half().double()
    return (q * d).reshape(v.shape)


def _silu(g):
    return g / (1 + torch.exp(-g))


def _dense(qd):
    q, d = qd
    return ((q.double() - 8) * d.double().unsqueeze(-1)).reshape(q.shape[0], -1)


def _exact_layer(case, seed, layer, x):
    H, I, E, k = SHAPES[case["shape"]]
    g = _norm(seed, case["shape"], layer).double()
    xn = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * g
    w, idx = torch.sort(xn @ _router(seed, case["shape"], layer, case["skew"])[0].double().T, dim=-1, descending=True, stable=True)
    w, idx = torch.softmax(w[:, :k], -1), idx[:, :k]
    xq, out = _q8(xn, 32, True), torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        t, j = torch.where(idx == e)
        gate, up, down = (_dense(m) for m in _pool_expert(seed, case["shape"], layer + e))
        h = _silu(xq[t] @ gate.T) * (xq[t] @ up.T)
        out.index_add_(0, t, (_q8(h, 32, True) @ down.T) * w[t, j].unsqueeze(-1))
    return out, idx.to(torch.int32), w


def _dense_q4k(b, rows):
    """Q4_K blocks -> [rows, cols] in 64 bits: y = d * scale * q - dmin * min per 32 values."""
    b = b.reshape(-1, 144)
    d = b[:, :4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].to(torch.int64)
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:12] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    q = b[:, 16:].reshape(-1, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
    return (d[:, :1, None] * sc[..., None] * q - d[:, 1:, None] * mn[..., None]).reshape(rows, -1)


def _exact_q4k_moe(case, seed, first, x):
    H, I, _, _ = SHAPES[case["shape"]]
    out, xq = torch.zeros(H, dtype=torch.float64, device="cuda"), _q8(x, 256, False)
    for e, w in enumerate(_expert_weights(case["experts"])):
        gate, up, down = _q4k_expert(seed, case["shape"], first + e).chunk(3)
        h = _silu(_dense_q4k(gate, I) @ xq) * (_dense_q4k(up, I) @ xq)
        out += float(w) * (_dense_q4k(down, H) @ _q8(h, 256, False))
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        out, idx, w = _exact_layer(case, seed, 0, _tokens(case, seed).double())
        return {"out": out, "idx": idx, "w": w}
    if kind == "stack":
        x = _tokens(case, seed).double()
        for l in range(case["layers"]):
            x = x + _exact_layer(case, seed, l, x)[0]
        return x
    if kind == "head":
        x, g = _randn(seed, 3, case["embed"]).double(), _randn(seed, 2, case["embed"], std=0.1, mean=1.0).double()
        xn = x / torch.sqrt((x * x).mean() + EPS) * g
        W = _randn(seed, 1, case["vocab"], case["embed"], std=0.02)
        y = torch.cat([c.double() @ xn for c in W.split(16384)])
        return {"logits": y, "token": int(y.argmax())}
    if kind == "sample":
        u = np.random.RandomState(int(seed) & 0x7FFFFFFF).random_sample(case["rows"])
        toks = []
        for r in range(case["rows"]):
            p = torch.softmax(_randn(seed, 1 + r, case["vocab"], std=2.5).double() / case["temperature"], 0)
            p, i = torch.sort(p, descending=True, stable=True)
            p = p[:int((p.cumsum(0) < case["top_p"]).sum()) + 1]
            c = p.cumsum(0) / p.sum()
            toks.append(int(i[min(int((c <= u[r]).sum()), p.numel() - 1)]))
        return toks
    if kind == "moe":
        return [_exact_q4k_moe(case, seed, c * case["experts"], _randn(seed, 400 + c, SHAPES[case["shape"]][0]).double())
                for c in range(case["calls"])]
    w, nrm, rope, kv, x = ([t.double() for t in v] if isinstance(v, list) else v.double() for v in _block_inputs(case, seed))
    n, hd, nh, nk = case["kv_len"], case["head_dim"], case["heads"], case["kv_heads"]

    def norm(v, g):
        return v / torch.sqrt((v * v).mean(-1, keepdim=True) + EPS) * g

    def rotate(v):
        a, b, c, s = v[:, :hd // 2], v[:, hd // 2:], rope[0][n], rope[1][n]
        return torch.cat([a * c - b * s, a * s + b * c], 1)

    xn = norm(x, nrm[0])
    q, kv[0][:, n] = rotate(norm((w[0] @ xn).reshape(nh, hd), nrm[2])), rotate(norm((w[1] @ xn).reshape(nk, hd), nrm[3]))
    kv[1][:, n] = (w[2] @ xn).reshape(nk, hd)
    K, V = (t[:, :n + 1].repeat_interleave(nh // nk, 0) for t in kv)
    p = torch.softmax((K @ q.unsqueeze(-1)).squeeze(-1) / math.sqrt(hd), -1)
    x = x + w[3] @ (p.unsqueeze(1) @ V).reshape(-1)
    return {"x": x + _exact_q4k_moe(case, seed, 0, norm(x, nrm[1])), "k": kv[0], "v": kv[1]}
