"""Performance cases of the routed-expert MoE step.

Each case is a stretch of a program's MoE work through the public binding
(nmoe_hip.Context over the C ABI): single-token decode over the layers of a
token, small and batched decode, chunked prompts and whole prefills, routing
alone; q4 and q2 experts, bf16 and q4 routers, bf16 and fp32 activations, with
and without the shared expert.  Hidden 2048, expert FFN 512, 256 experts and
group 64 are the format's constants.

A case is a dict of
  call    "layer"  [shared_expert +] moe_layer per layer (routing included)
          "block"  moe_block per layer (norms, q4 router, shared expert; 1 token)
          "stack"  one moe_stack over all layers (1 token)
          "logits" experts_from_logits per layer (router logits already there)
          "route"  route per layer (router logits and top-k only)
  bits    4 or 2: the experts' code width
  k       experts a token
  tokens  tokens of a call
  x       "bf16" or "f32" activations
  router  "bf16" or "q4" ("none" where the logits are given)
  load    "even" or "zipf": how the given logits spread tokens over experts
  shared  whether the shared expert runs too
  layers  layers a pass goes through, each with its own weights, residual and
          input, as a token's way through the model touches them: a pass that
          repeated one layer would find its experts in the memory-side cache
"""
import math
import os
import sys

import numpy as np
import torch

# torch brings the HIP runtime the library then shares (same soname), so both
# use the same device pointers and streams
_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "nano-metal-moe-qwen36_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import nmoe_hip as nh  # noqa: E402

H, F, E, G = nh.HIDDEN, nh.INTER, nh.EXPERTS, nh.GROUP
SIGMA = {4: 0.02, 2: 0.05}  # expert scales, as bench.py's synthetic layers
EPS = 1e-6
MAX_TOKENS = 4096
_stream = None


def _case(name, call, bits, k, tokens, x, router, shared, layers, load="even"):
    return {"name": name, "call": call, "bits": bits, "k": k, "tokens": tokens, "x": x, "router": router,
            "load": load, "shared": shared, "layers": layers}


def listed():
    return [
        # one decode token, layer by layer, as the runtime's expert tail calls it
        _case("decode_q4", "layer", 4, 8, 1, "bf16", "bf16", False, 24),
        # the same with the smaller packs and fewer experts
        _case("decode_q2_k6", "layer", 2, 6, 1, "f32", "bf16", False, 24),
        # one decode token through whole MoE halves: norms, q4 router, shared expert
        _case("block_q4", "block", 4, 8, 1, "f32", "q4", True, 20),
        # a token's 40 layers in one call
        _case("stack_q4", "stack", 4, 8, 1, "f32", "bf16", False, 40),
        # a handful of sequences decoding together, the model's own tensors
        _case("batch4_shared_q4", "layer", 4, 8, 4, "f32", "q4", True, 6),
        # a ragged small batch
        _case("batch13_q2", "layer", 2, 8, 13, "bf16", "bf16", False, 4),
        # batched decode with skewed experts, logits at hand
        _case("batch64_zipf_q4", "logits", 4, 8, 64, "bf16", "none", False, 2, "zipf"),
        # a prompt chunk, the model's own tensors, odd length
        _case("chunk251_shared_q4", "layer", 4, 8, 251, "f32", "q4", True, 1),
        # a middle-sized prompt with q2 experts
        _case("prefill1000_shared_q2", "layer", 2, 8, 1000, "bf16", "bf16", True, 1),
        # a 2048-token prefill's experts, logits at hand
        _case("prefill2048_q4", "logits", 4, 8, 2048, "bf16", "none", False, 1),
        # routing of a prompt on its own (placement, statistics)
        _case("route3001", "route", 4, 8, 3001, "bf16", "bf16", False, 1),
        # the largest: a long prompt through the whole MoE half, the model's own tensors
        _case("prefill4096_shared_q4", "layer", 4, 8, 4096, "f32", "q4", True, 1),
    ]


def draw(rng):
    call = rng.choice(["layer", "layer", "layer", "layer", "logits", "logits", "block", "stack", "route"])
    bits, k = rng.choice([4, 4, 2]), rng.choice([8, 8, 8, 6, rng.randint(1, 7)])
    x, router, shared = rng.choice(["bf16", "f32"]), rng.choice(["bf16", "q4"]), rng.random() < 0.5
    if call in ("block", "stack"):
        layers = rng.randint(12, 20) if call == "block" else rng.randint(8, 40)
        return _pure(call, bits, k, 1, "f32", "q4" if call == "block" else router, call == "block", layers)
    tokens = min(MAX_TOKENS, int(math.exp(rng.uniform(0.0, math.log(MAX_TOKENS + 1.0)))))
    if call == "route":
        return _pure(call, bits, k, tokens, x, router, False, 1)
    # as many layers as keep a pass's experts beyond the 256 MB memory-side cache
    layers = max(1, min(24, int(340e6 / (nh.EXPERT_SIZE[bits] * E * (1 - (1 - k / E) ** tokens)))))
    if call == "logits":
        return _pure(call, bits, k, tokens, x, "none", False, layers, rng.choice(["even", "zipf"]))
    return _pure(call, bits, k, tokens, x, router, shared, layers)


def _pure(*a):
    c = _case("", *a)
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs

def _gen(case, seed, layer):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + layer * 8191 + case["tokens"] * 31 + case["bits"]) & 0x7FFFFFFFFFFF)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _q4(g, rows, cols, sigma):
    """A q4 tensor as the model stores it: codes, bf16 scales, biases -8 * scale."""
    w = torch.randint(-2 ** 31, 2 ** 31, (rows, cols // 8), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    s = (_randn(g, rows, cols // G) * sigma).to(torch.bfloat16)
    return w, s, (-8.0 * s.float()).to(torch.bfloat16)


def _inputs(case, seed, layer):
    """One layer's inputs and tensors, from the seed alone."""
    g, T = _gen(case, seed, layer), case["tokens"]
    d = {"h": _randn(g, T, H)}
    if case["call"] in ("layer", "logits", "route"):
        # normalised hidden states share a direction, which skews the experts' loads
        x = _randn(g, T, H) + (0.6 * _randn(g, 1, H) if T > 1 else 0.0)
        x = x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + EPS)
        d["x"] = x.to(torch.bfloat16) if case["x"] == "bf16" else x
    if case["router"] == "bf16":
        d["router"] = (0.02 * _randn(g, E, H)).to(torch.bfloat16)
    elif case["router"] == "q4":
        d["router"] = _q4(g, E, H, 0.004)
    elif case["load"] == "zipf":  # ln p_e + Gumbel, p_e ~ rank^-1.1 over shuffled experts
        rank = torch.randperm(E, generator=g, device="cuda") + 1
        u = torch.rand(T, E, generator=g, device="cuda").clamp(1e-7, 1 - 1e-7)
        d["logits"] = -1.1 * torch.log(rank.float()) - torch.log(-torch.log(u))
    else:
        d["logits"] = torch.rand(T, E, generator=g, device="cuda")
    if case["shared"]:
        d["se"] = [_q4(g, F, H, 0.004), _q4(g, F, H, 0.004), _q4(g, H, F, 0.008), _q4(g, 1, H, 0.004)]
    if case["call"] == "block":
        d["norms"] = [(0.1 * _randn(g, H)).to(torch.bfloat16) for _ in range(2)]
    return d


class _State:
    """The context (with its resident layers), inputs and outputs of one case; gives the device memory back when dropped."""

    def __init__(self, case, seed):
        global _stream
        if _stream is None:
            _stream = torch.cuda.Stream()  # the program's one stream: a context's launches stay ordered
        self.case, self.stream = case, _stream.cuda_stream
        T, n = case["tokens"], case["layers"]
        self.ctx = nh.Context(torch.cuda.current_device(), max_tokens=T)
        self.d = [_inputs(case, seed, l) for l in range(n)]
        if case["call"] != "route":
            for l in range(n):
                self.ctx.synth_layer(l, case["bits"], int(seed), SIGMA[case["bits"]])
        self.xdt = nh.BF16 if case["x"] == "bf16" else nh.F32
        f32 = dict(device="cuda", dtype=torch.float32)
        self.out = torch.zeros(n, T, H, **f32)
        self.idx = torch.zeros(n, T, nh.MAX_K, device="cuda", dtype=torch.int32)
        self.w = torch.zeros(n, T, nh.MAX_K, **f32)
        self.p = []  # per layer: the pointers its calls take
        p = lambda t: t.data_ptr()
        for l, d in enumerate(self.d):
            q = {"out": p(self.out[l]), "idx": p(self.idx[l]), "w": p(self.w[l]), "h": p(d["h"])}
            q["x"] = p(d["x"]) if "x" in d else None
            if case["router"] == "bf16":
                q["router"] = nh.Context.router_bf16(p(d["router"]))
            elif case["router"] == "q4":
                q["router"] = nh.Context.router_q4(*(p(t) for t in d["router"]))
            else:
                q["logits"] = p(d["logits"])
            if case["shared"]:
                q["se"] = nh.Context.shared_expert_desc(*([p(t) for t in s] for s in d["se"]))
            if case["call"] == "block":
                q["blk"] = nh.MoeBlock(q["router"], 1, q["se"], p(d["norms"][0]), p(d["norms"][1]), 1, EPS)
            self.p.append(q)
        if case["call"] == "layer" and case["shared"]:
            self.so, self.sg = torch.zeros(n, T, H, **f32), torch.zeros(n, T, **f32)
        if case["call"] == "route":
            self.logits = torch.zeros(n, T, E, **f32)
        if case["call"] == "block":
            self.nx = torch.zeros(n, T, H, **f32)
        if case["call"] == "stack":
            self.h_seq = torch.zeros(n + 1, H, **f32)
            self.h_seq[0] = self.d[0]["h"][0]
            self.routers = [q["router"] for q in self.p]
        torch.cuda.synchronize()

    def __del__(self):
        if getattr(self, "ctx", None) is not None:
            self.ctx.close()


def prepare(case, seed):
    return _State(case, seed)


def run(st):
    c, ctx, s = st.case, st.ctx, st.stream
    call, k, T = c["call"], c["k"], c["tokens"]
    if call == "stack":
        ctx._check(ctx.moe_stack(range(c["layers"]), st.routers, k, EPS, st.h_seq.data_ptr(), st.idx.data_ptr(),
                                 st.w.data_ptr(), stream=s))
        return {"h": st.h_seq, "idx": st.idx, "w": st.w}
    for l, p in enumerate(st.p):
        if call == "layer":
            so = sg = None
            if c["shared"]:
                so, sg = st.so[l].data_ptr(), st.sg[l].data_ptr()
                ctx._check(ctx.shared_expert(p["se"], p["x"], st.xdt, T, so, sg, stream=s))
            ctx._check(ctx.moe_layer(l, p["router"], p["x"], st.xdt, T, k, p["h"], p["out"], p["idx"], p["w"],
                                     shared_out=so, shared_gate_raw=sg, stream=s))
        elif call == "logits":
            ctx._check(ctx.experts_from_logits(l, p["logits"], p["x"], st.xdt, T, k, p["h"], p["out"], p["idx"],
                                               p["w"], stream=s))
        elif call == "block":
            ctx._check(ctx.moe_block(l, p["blk"], p["h"], k, p["out"], st.nx[l].data_ptr(), p["idx"], p["w"],
                                     stream=s))
        else:
            ctx._check(ctx.route(p["router"], p["x"], st.xdt, T, k, p["idx"], p["w"], st.logits[l].data_ptr(),
                                 stream=s))
    r = {"idx": st.idx, "w": st.w}
    if call == "route":
        return {**r, "logits": st.logits}
    r["out"] = st.out
    if call == "block":
        r["next_x"] = st.nx
    elif c["shared"]:
        r["shared_out"], r["shared_gate_raw"] = st.so, st.sg
    return r


# ------------------------------------------------------------------ work

def _experts_met(case):
    """About how many distinct experts a layer's tokens select."""
    T, k = case["tokens"], case["k"]
    if T == 1:
        return k
    r = np.random.default_rng(1)
    if case["router"] == "none":
        lg = r.gumbel(size=(T, E)) - 1.1 * np.log(np.arange(1, E + 1)) if case["load"] == "zipf" else r.random((T, E))
    else:
        lg = r.standard_normal((T, E)) + 0.6 * r.standard_normal((1, E))
    return len(np.unique(np.argpartition(-lg, k - 1, axis=1)[:, :k]))


def _q4_bytes(rows, cols):
    return rows * cols // 2 + 2 * (rows * cols // G) * 2


def work(case):
    T, k, call = case["tokens"], case["k"], case["call"]
    xb = 2 if case["x"] == "bf16" else 4
    b = T * 64  # idx, w
    f = 0.0
    if case["router"] == "none":
        b += T * E * 4
    else:
        b += E * H * 2 if case["router"] == "bf16" else _q4_bytes(E, H)
        f += 2.0 * T * E * H
    if call == "route":
        b += T * (H * xb + E * 4)
    else:
        b += _experts_met(case) * nh.EXPERT_SIZE[case["bits"]]
        b += T * H * (4 if call in ("block", "stack") else xb + 4)  # x and h_mid, or h_mid alone
        b += T * H * 4  # out
        f += 2.0 * T * k * 3 * H * F
        if case["shared"]:
            b += 2 * _q4_bytes(F, H) + _q4_bytes(H, F) + _q4_bytes(1, H)
            f += 2.0 * T * (3 * H * F + H)
            if call == "layer":
                b += T * (H + 1) * 4  # shared_out, shared_gate_raw
        if call == "block":
            b += 2 * H * 2 + H * 4  # norm weights, next_x
    return {"bytes": float(b * case["layers"]), "flops": f * case["layers"]}


def tolerance(case):
    """About four times the error seen against exact()."""
    if case["call"] == "stack":  # rounding travels through its layers
        return {"rel": 2e-5, "max": 1e-3, "differ": 0.0}
    if case["tokens"] < 8 or case["call"] == "route":  # fp32 throughout
        return {"rel": 2e-6, "max": 1e-4, "differ": 0.0}
    # the grouped calls' activations carry 16 mantissa bits (two bf16 parts),
    # and their codes an offset of 128 that cancels (more so for q2's 0..3)
    return {"rel": 1e-4, "max": 4e-3, "differ": 0.0}


# ----------------------------------------------------------------- exact

_M64 = (1 << 64) - 1
_GOLD, _C1, _C2 = 0x9E3779B97F4A7C15, 0xBF58476D1CE4E5B9, 0x94D049BB133111EB


def _signed(v):
    v &= _M64
    return v - (1 << 64) if v >> 63 else v


def _mix(z):
    """SplitMix64's finaliser, on a Python integer or an int64 tensor."""
    if isinstance(z, int):
        z = ((z ^ (z >> 30)) * _C1) & _M64
        z = ((z ^ (z >> 27)) * _C2) & _M64
        return z ^ (z >> 31)
    shr = lambda v, n: (v >> n) & ((1 << (64 - n)) - 1)
    z = (z ^ shr(z, 30)) * _signed(_C1)
    z = (z ^ shr(z, 27)) * _signed(_C2)
    return z ^ shr(z, 31)


def _rand64(seed, layer, expert, tag, n, device):
    stream = _mix(_mix((seed + _GOLD) & _M64) ^ ((layer << 40) | (expert << 16) | tag))
    return _mix((torch.arange(1, n + 1, dtype=torch.int64, device=device) * _signed(_GOLD)) + _signed(stream))


def _expert64(bits, seed, layer, expert, device="cuda"):
    """gate, up [512][2048] and down [2048][512] of a synthetic expert, dequantised in 64 bits."""
    ws, vpw = [], 32 // bits
    shifts = torch.arange(vpw, dtype=torch.int64, device=device) * bits
    for m, (rows, cols) in enumerate(((F, H), (F, H), (H, F))):
        words = _rand64(seed, layer, expert, 2 * m, rows * cols // vpw // 2, device).view(torch.int32)
        q = (words.to(torch.int64)[:, None] >> shifts) & ((1 << bits) - 1)
        r = _rand64(seed, layer, expert, 2 * m + 1, 3 * rows * cols // G, device).view(-1, 3)
        u = sum((r >> s) & 0xFFFF for s in (0, 16, 32, 48)).sum(dim=1)
        normal = (u + 6).to(torch.float32) * (1.0 / 65536.0) - 6.0
        s = (normal * torch.tensor(SIGMA[bits], dtype=torch.float32, device=device)).to(torch.bfloat16).float()
        b = ((-8.0 if bits == 4 else -1.5) * s).to(torch.bfloat16)
        w = q.view(rows, cols // G, G).double() * s.double().view(rows, -1, 1) + b.double().view(rows, -1, 1)
        ws.append(w.view(rows, cols))
    return ws


def _deq64(t):
    w, s, b = t
    shifts = torch.arange(8, dtype=torch.int64, device=w.device) * 4
    q = ((w.to(torch.int64)[..., None] >> shifts) & 15).view(s.shape[0], s.shape[1], G)
    return (q.double() * s.double()[..., None] + b.double()[..., None]).view(s.shape[0], -1)


def _route64(logits, k):
    p, i = torch.sort(torch.softmax(logits, dim=1), dim=1, descending=True, stable=True)
    p, i = p[:, :k], i[:, :k]
    return p / p.sum(dim=1, keepdim=True), i


def _pad(w):
    return torch.nn.functional.pad(w, (0, nh.MAX_K - w.shape[1]))


def _experts64(case, seed, layer, x, w, i):
    y = torch.zeros(x.shape[0], H, dtype=torch.float64, device=x.device)
    for e in torch.unique(i).tolist():
        t, s = (i == e).nonzero(as_tuple=True)
        gate, up, down = _expert64(case["bits"], int(seed), layer, e, x.device)
        xe = x[t]
        a = torch.nn.functional.silu(xe @ gate.T) * (xe @ up.T)
        y.index_add_(0, t, w[t, s, None] * (a @ down.T))
    return y


def _norm64(h, wt=None):
    x = h / torch.sqrt(h.square().mean(dim=1, keepdim=True) + EPS)
    return x if wt is None else x * (1.0 + wt.double())


def exact(case, seed):
    out = {"idx": None, "w": []}
    put = lambda key, v: out.setdefault(key, []).append(v)
    call, k = case["call"], case["k"]
    h = None
    for l in range(case["layers"]):
        d = _inputs(case, seed, l)
        if call == "stack":
            if h is None:
                h = d["h"].double()
                put("h", h[0])
        else:
            h = d["h"].double()
        if call == "block":
            x = _norm64(h, d["norms"][0])
        else:
            x = _norm64(h) if call == "stack" else d["x"].double()
        if "logits" in d:
            lg = d["logits"].double()
        else:
            lg = x @ (_deq64(d["router"]) if case["router"] == "q4" else d["router"].double()).T
        w, i = _route64(lg, k)
        put("w", _pad(w))
        if call == "route":
            put("logits", lg)
            continue
        y = h + _experts64(case, seed, l, x, w, i)
        if case["shared"]:
            gate, up, down, score = (_deq64(t) for t in d["se"])
            so = (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T
            sg = (x @ score.T)[:, 0]
            y = y + torch.sigmoid(sg)[:, None] * so
            if call == "layer":
                put("shared_out", so)
                put("shared_gate_raw", sg)
        if call == "stack":
            h = y
            put("h", h[0])
        else:
            put("out", y)
            if call == "block":
                put("next_x", _norm64(y, d["norms"][1]))
    return {key: None if v is None else torch.stack(v) for key, v in out.items()}
