"""The calls that a program on this framework makes, as timed cases.

A case is a dict of plain values.  `kind` says which entry point it goes through:

  layer    one MoE layer on device activations, `Backend.moe_forward` (a decode step of S
           streams, or a prefill of S tokens): router, gate, top-k, experts, combine, shared
           expert, residual
  stack    a decode step of a small stack, `DeviceStack.step`: for each layer the RMSNorm and
           the MoE layer on the residual, then the final norm, the bf16 head and the pick
  group    the grouped experts of an engine that routes by itself, host activations and
           host-made groups, `Backend.moe_group`
  matmul   an engine's dense projection on host activations, `Backend.matmul_*`
  glm      the expert groups of the GLM engine's table on host rows, `Coli.expert_group`
  router   the GLM engine's device router on one row, `Coli.router`

Weights are N(0, 0.02) quantised to int4 (one f32 scale per `gs` inputs, or per row for
gs = 0) or rounded to bf16, activations N(0, 1), the workload of the benchmark's
configurations (`sabrewing_amd/configs.py`).  Everything is made on the device from the seed.
"""
import math

import numpy as np
import torch

from sabrewing_amd import configs as cf
from sabrewing_amd.backend import Backend, DeviceLayer, desc_of
from sabrewing_amd.coli import Coli
from sabrewing_amd.stack import DeviceStack, NORM_EPS

SIGMA = cf.WEIGHT_SIGMA
_handles = {}


def _be():
    if "be" not in _handles:
        _handles["be"] = Backend(0)
    return _handles["be"]


def _coli():
    if "coli" not in _handles:
        _handles["coli"] = Coli([0])
    return _handles["coli"]


# ------------------------------------------------------------------ cases ----

def _layer(name, cfg, S, **kw):
    d = dict(name=name, kind="layer", S=S, D=cfg.D, E=cfg.E, K=cfg.K, I=cfg.I, Is=cfg.Is, act=cfg.route_act,
             corr=cfg.use_corr_bias, norm=cfg.norm_topk, scale=cfg.route_scale, shared=cfg.shared_mode, gs=cfg.gs,
             router_bf16=bool(cfg.router_bf16), x_bf16=bool(cfg.x_bf16), n_shared=cfg.n_shared)
    d.update(kw)
    return d


def listed():
    return [
        # one stream decoding: the smallest call, three dependent launches
        _layer("c2_decode_1", cf.C2, 1),
        # a server's decode batches, few streams to many
        _layer("c2_decode_8", cf.C2, 8),
        _layer("c2_decode_32", cf.C2, 32),
        _layer("c2_decode_64", cf.C2, 64),
        # a short prompt, or a wide batch of decoding streams: an odd count between decode and prefill
        _layer("c2_mixed_181", cf.C2, 181),
        # the benchmark's prefill: the largest call
        _layer("c2_prefill_2048", cf.C2, 2048),
        # the small model: f32 router, softmax, no shared expert, a ragged prompt
        _layer("c1_prefill_333", cf.C1, 333),
        # the stack's decode step (two of its layers) through the norms, the head and the pick
        dict(name="c5_stack_8", kind="stack", S=8, layers=2, D=cf.C5_LAYER.D, E=cf.C5_LAYER.E, K=cf.C5_LAYER.K,
             I=cf.C5_LAYER.I, V=cf.C5_VOCAB),
        # the Laguna engine's grouped hook: per-row int4, a chunk of 128 rows, host activations
        dict(name="laguna_group_128", kind="group", S=128, D=cf.C2.D, E=cf.C2.E, K=cf.C2.K, I=cf.C2.I, gs=0),
        # an engine's dense bf16 projection on a small batch of host rows
        dict(name="matmul_bf16_16", kind="matmul", weights="bf16", S=16, I=4096, O=4096, gs=0),
        # the GLM engine's decode: eight experts, one row each, three tensors per expert
        dict(name="glm_decode_8x1", kind="glm", experts=8, rows=1, D=5120, I=1536, gs=0),
        # the Inkling layer: f32 router with shared gates, per-row int4, two gated bf16 shared experts
        _layer("inkling_4", cf.INKLING, 4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer"] * 8 + ["stack", "group", "group", "matmul", "matmul", "glm", "glm", "router"])
    if kind == "layer":
        cfg = rng.choice([cf.C2, cf.C2, cf.C2_SIGMOID, cf.C2_SQRTSP, cf.C1, cf.C1_OLMOE, cf.QWEN, cf.C5_LAYER, cf.INKLING])
        S = _log_int(rng, 1, 64 if cfg is cf.INKLING else 1024 if cfg is cf.C5_LAYER else 2048)
        c = _layer(None, cfg, S)
        del c["name"]
        if rng.random() < 0.4:                    # another layer shape of the same contract
            c["D"] = 128 * rng.randint(4, cfg.D // 128)
            c["I"] = 128 * rng.randint(2, cfg.I // 128)
            c["Is"] = c["I"] if cfg.Is else 0
            c["E"] = rng.randint(max(cfg.K, 16), cfg.E)
            if cfg is not cf.INKLING:
                c["gs"] = rng.choice([0, 32, 32, 64, 128])
        return c
    if kind == "stack":
        return dict(kind="stack", S=rng.randint(1, 32), layers=rng.randint(1, 2), D=cf.C5_LAYER.D, E=cf.C5_LAYER.E,
                    K=cf.C5_LAYER.K, I=128 * rng.randint(4, cf.C5_LAYER.I // 128), V=4 * rng.randint(4000, cf.C5_VOCAB // 4))
    if kind == "group":
        return dict(kind="group", S=_log_int(rng, 1, 256), D=128 * rng.randint(8, 32), E=rng.randint(16, 256),
                    K=rng.randint(1, 10), I=128 * rng.randint(2, 12), gs=rng.choice([0, 0, 32, 128]))
    if kind == "matmul":
        w = rng.choice(["bf16", "bf16", "bf16_rx", "q8", "q4", "q4"])
        return dict(kind="matmul", weights=w, S=_log_int(rng, 1, 64), I=32 * rng.randint(16, 160), O=rng.randint(256, 6144),
                    gs=rng.choice([0, 32]) if w == "q4" else 0)
    if kind == "glm":
        return dict(kind="glm", experts=rng.randint(1, 16), rows=_log_int(rng, 1, 96), D=128 * rng.randint(8, 40),
                    I=128 * rng.randint(4, 12), gs=rng.choice([0, 0, 64]))
    return dict(kind="router", D=32 * rng.randint(32, 160), E=rng.randint(32, 256), K=rng.randint(2, 8))


# ----------------------------------------------------------------- inputs ----

class _Dev:
    """A torch tensor handed to the framework as device memory."""

    def __init__(self, t):
        self.t = t

    def __int__(self):
        return self.t.data_ptr()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, sigma=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * sigma


def _q4(g, rows, K, gs):
    """packed int4 [rows, K/2] (low nibble: the even input, offset 8) and f32 scales [rows, K/gs] (or [rows, 1])"""
    n = gs if gs > 0 else K
    q = torch.empty(rows, K // 2, dtype=torch.uint8, device="cuda")
    s = torch.empty(rows, K // n, dtype=torch.float32, device="cuda")
    step = max(1, (1 << 26) // K)
    for r in range(0, rows, step):
        m = min(step, rows - r)
        w = _randn(g, m, K // n, n, sigma=SIGMA)
        sc = w.abs().amax(2) / 7
        v = ((w / sc[:, :, None]).round_().clamp_(-8, 7) + 8).to(torch.uint8).view(m, K // 2, 2)
        q[r:r + m] = v[:, :, 0] | (v[:, :, 1] << 4)
        s[r:r + m] = sc
    return q, s


def _unq4(q, s):
    """the weights of rows of _q4 in 64 bits"""
    v = torch.stack([q & 15, q >> 4], dim=2).view(q.shape[0], -1).to(torch.float64) - 8
    return (v.view(q.shape[0], s.shape[1], -1) * s.to(torch.float64)[:, :, None]).view(q.shape[0], -1)


def _cfg(c):
    return cf.MoeConfig("case", D=c["D"], E=c["E"], K=c["K"], I=c["I"], Is=c["Is"], route_act=c["act"],
                        use_corr_bias=c["corr"], norm_topk=c["norm"], route_scale=c["scale"], shared_mode=c["shared"],
                        gs=c["gs"], router_bf16=c["router_bf16"], x_bf16=c["x_bf16"], n_shared=c["n_shared"])


def _stack_cfg(c):
    return cf.scaled(cf.C5_LAYER, D=c["D"], E=c["E"], K=c["K"], I=c["I"], name="case")


def _weights(g, cfg):
    """a layer's tensors as torch makes them"""
    D, I, Is, E = cfg.D, cfg.I, cfg.Is, cfg.E
    w = {"router": _randn(g, cfg.router_rows, D, sigma=SIGMA)}
    if cfg.router_bf16:
        w["router"] = w["router"].to(torch.bfloat16)
    w["gu_q"], w["gu_s"] = _q4(g, E * 2 * I, D, cfg.gs)
    w["dn_q"], w["dn_s"] = _q4(g, E * D, I, cfg.gs)
    if cfg.use_corr_bias:
        w["corr_bias"] = _randn(g, E, sigma=0.01)
    ns = cfg.n_shared_experts
    if ns:
        w["sg"] = _randn(g, ns * Is, D, sigma=SIGMA).to(torch.bfloat16)
        w["su"] = _randn(g, ns * Is, D, sigma=SIGMA).to(torch.bfloat16)
        w["sd"] = _randn(g, ns * D, Is, sigma=SIGMA).to(torch.bfloat16)
    return w


def _rows(g, S, D, bf16):
    x = _randn(g, S, D)
    return x.to(torch.bfloat16).float() if bf16 else x


def _chained(be, W):
    """a router or head [R, D] in the order the routing kernels stream"""
    R, D = W.shape
    out = torch.empty((R + 3) // 4 * 4 * D, dtype=W.dtype, device="cuda")
    torch.cuda.synchronize()
    be.check(be.lib.lag_hip_router_chain(W.data_ptr(), out.data_ptr(), R, D, int(W.dtype == torch.bfloat16)), "router chain")
    be.sync()
    return _Dev(out)


def _device_layer(be, cfg, w):
    dl = DeviceLayer(be, cfg)
    dl.router = _chained(be, w["router"])
    for k in ("gu_q", "gu_s", "dn_q", "dn_s", "corr_bias", "sg", "su", "sd"):
        if k in w:
            setattr(dl, k, _Dev(w[k]))
    return dl


def _groups(c, seed):
    """the groups an engine makes from its own routing: K distinct experts per row, sorted by expert"""
    r = np.random.default_rng([int(seed), 17])
    S, E, K = c["S"], c["E"], c["K"]
    sel = np.argsort(r.random((S, E)), axis=1)[:, :K].astype(np.int32)
    wts = r.random((S, K)).astype(np.float32) + np.float32(0.1)
    wts = (wts / wts.sum(1, keepdims=True)).astype(np.float32)
    order = np.argsort(sel.reshape(-1), kind="stable")
    gexp, gcnt = np.unique(sel, return_counts=True)
    gbeg = np.concatenate([[0], np.cumsum(gcnt)[:-1]])
    rowof = np.empty(S * K, np.int32)
    rowof[order] = np.arange(S * K, dtype=np.int32)
    i32 = lambda a: np.ascontiguousarray(a, np.int32)
    return sel, wts, i32(gexp), i32(gbeg), i32(gcnt), i32(order // K), rowof


def _inputs(c, seed):
    g, kind = _gen(seed), c["kind"]
    if kind == "layer":
        cfg = _cfg(c)
        w = _weights(g, cfg)
        return cfg, w, _rows(g, c["S"], cfg.D, cfg.x_bf16), _randn(g, c["S"], cfg.D)
    if kind == "stack":
        cfg = _stack_cfg(c)
        ws = [_weights(g, cfg) for _ in range(c["layers"])]
        norms = 1.0 + _randn(g, c["layers"] + 1, cfg.D, sigma=SIGMA)
        head = _randn(g, c["V"], cfg.D, sigma=SIGMA).to(torch.bfloat16)
        return cfg, ws, norms, head, _rows(g, c["S"], cfg.D, True)
    if kind == "group":
        gu, dn = _q4(g, c["E"] * 2 * c["I"], c["D"], c["gs"]), _q4(g, c["E"] * c["D"], c["I"], c["gs"])
        return gu, dn, _randn(g, c["S"], c["D"]).cpu().numpy(), _groups(c, seed)
    if kind == "matmul":
        I, O, x = c["I"], c["O"], _randn(g, c["S"], c["I"]).cpu().numpy()
        if c["weights"].startswith("bf16"):
            return (_randn(g, O, I, sigma=SIGMA).to(torch.bfloat16),), x
        if c["weights"] == "q8":
            w = _randn(g, O, I, sigma=SIGMA)
            s = w.abs().amax(1) / 127
            return ((w / s[:, None]).round().clamp(-127, 127).to(torch.int8), s), x
        return _q4(g, O, I, c["gs"]), x
    if kind == "glm":
        e, D, I = c["experts"], c["D"], c["I"]
        ts = [(_q4(g, I, D, c["gs"]), _q4(g, I, D, c["gs"]), _q4(g, D, I, c["gs"])) for _ in range(e)]
        return ts, _randn(g, e * c["rows"], D).cpu().numpy()
    return _randn(g, c["E"], c["D"], sigma=SIGMA), _randn(g, c["E"], sigma=0.01), _randn(g, c["D"])


class _State:
    def __init__(self, **kw):
        self.tensors = []                         # the GLM table's tensors, given back with the state
        self.__dict__.update(kw)

    def __del__(self):
        for t in self.tensors:
            t.free()


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "layer":
        be = _be()
        cfg, w, x, res = _inputs(c, seed)
        dl = _device_layer(be, cfg, w)
        s = _State(be=be, dl=dl, desc=desc_of(cfg), w=dl.weights(), x=_Dev(x), out=_Dev(res), S=c["S"])
    elif kind == "stack":
        be = _be()
        cfg, ws, norms, head, x = _inputs(c, seed)
        st = DeviceStack(be, cfg, c["V"])
        st.layers = [_device_layer(be, cfg, w) for w in ws]
        st.norms = [_Dev(norms[i]) for i in range(c["layers"])]
        st.final_norm = _Dev(norms[c["layers"]])
        st.head = _chained(be, head)
        h, xn = torch.empty_like(x), torch.empty_like(x)
        logits = torch.empty(c["S"], c["V"], device="cuda")
        tok = torch.empty(c["S"], dtype=torch.int32, device="cuda")
        s = _State(be=be, st=st, x=x, h=_Dev(h), xn=_Dev(xn), logits=_Dev(logits), tok=_Dev(tok), S=c["S"])
    elif kind == "group":
        gu, dn, x, (_, wts, gexp, gbeg, gcnt, grow, rowof) = _inputs(c, seed)
        L = _State(D=c["D"], I=c["I"], gu_q=_Dev(gu[0]), gu_s=_Dev(gu[1]), dn_q=_Dev(dn[0]), dn_s=_Dev(dn[1]))
        s = _State(be=_be(), L=L, x=x, args=(gexp, gbeg, gcnt, grow, rowof, wts), K=c["K"], gs=c["gs"])
    elif kind == "matmul":
        W, x = _inputs(c, seed)
        s = _State(be=_be(), W=[_Dev(t) for t in W], x=x, weights=c["weights"], O=c["O"], gs=c["gs"])
    elif kind == "glm":
        co = _coli()
        ts, x = _inputs(c, seed)
        D, I, gs = c["D"], c["I"], c["gs"]
        up = [[co.upload(q.cpu().numpy(), sc.cpu().numpy(), k, o, gs=gs) for (q, sc), k, o in zip(t, (D, D, I), (I, I, D))]
              for t in ts]
        s = _State(co=co, g=[t[0] for t in up], u=[t[1] for t in up], d=[t[2] for t in up], rows=[c["rows"]] * c["experts"],
                   x=x, tensors=[t for e in up for t in e])
    else:
        W, b, x = _inputs(c, seed)
        s = _State(co=_coli(), W=_Dev(W), b=_Dev(b), x=_Dev(x), D=c["D"], E=c["E"], K=c["K"])
    s.kind = kind
    torch.cuda.synchronize()
    return s


def run(s):
    if s.kind == "layer":                         # the residual rows take the layer's update, as in a decode loop
        s.be.moe_forward(s.desc, s.w, s.x, s.out, s.S)
        return s.out.t
    if s.kind == "stack":
        s.be.check(s.be.lib.lag_hip_d2d(int(s.h), s.x.data_ptr(), s.x.numel() * 4), "d2d")
        s.st.step(s.h, s.xn, s.logits, s.tok, s.S)
        return {"h": s.h.t, "logits": s.logits.t}
    if s.kind == "group":
        return s.be.moe_group(s.x, s.L, *s.args, s.K, s.gs)
    if s.kind == "matmul":
        if s.weights == "bf16":
            return s.be.matmul_bf16(s.x, s.W[0], s.O)
        if s.weights == "bf16_rx":
            return s.be.matmul_bf16_rx(s.x, s.W[0], s.O)
        if s.weights == "q8":
            return s.be.matmul_q8(s.x, s.W[0], s.W[1], s.O)
        return s.be.matmul_q4(s.x, s.W[0], s.W[1], s.O, s.gs)
    if s.kind == "glm":
        return s.co.expert_group(s.g, s.u, s.d, s.rows, s.x)
    idx, w, _ = s.co.router(0, int(s.x), int(s.W), int(s.b), s.D, s.E, s.K)
    return {"idx": idx, "w": w}


# ------------------------------------------------------------------- work ----

def _distinct(E, S, K):
    """expected distinct experts of S rows of K distinct uniform picks"""
    return E * (1.0 - (1.0 - K / E) ** S)


def work(case):
    c, kind = case, case["kind"]
    if kind == "layer":
        cfg = _cfg(c)
        return {"bytes": cfg.step_bytes(c["S"], _distinct(cfg.E, c["S"], cfg.K)), "flops": cfg.flops(c["S"])}
    if kind == "stack":
        cfg, S = _stack_cfg(c), c["S"]
        layer = cfg.step_bytes(S, _distinct(cfg.E, S, cfg.K))
        return {"bytes": c["layers"] * layer + c["V"] * cfg.D * 2 + S * c["V"] * 4,
                "flops": c["layers"] * cfg.flops(S) + 2 * S * c["V"] * cfg.D}
    if kind == "group":
        S, D, I, K, n = c["S"], c["D"], c["I"], c["K"], _distinct(c["E"], c["S"], c["K"])
        sc = 4 * (2 * I * (D // c["gs"]) + D * (I // c["gs"])) if c["gs"] else 4 * (2 * I + D)
        return {"bytes": n * (3 * D * I / 2 + sc) + 2 * S * D * 4, "flops": 6 * S * K * D * I}
    if kind == "matmul":
        S, I, O = c["S"], c["I"], c["O"]
        b = {"bf16": 2, "bf16_rx": 2, "q8": 1, "q4": 0.5}[c["weights"]]
        sc = 0 if b == 2 else O * 4 * (I // c["gs"] if c["gs"] else 1)
        return {"bytes": O * I * b + sc + S * (I + O) * 4, "flops": 2 * S * I * O}
    if kind == "glm":
        e, T, D, I = c["experts"], c["experts"] * c["rows"], c["D"], c["I"]
        sc = 4 * (2 * I * (D // c["gs"]) + D * (I // c["gs"])) if c["gs"] else 4 * (2 * I + D)
        return {"bytes": e * (3 * D * I / 2 + sc) + 2 * T * D * 4, "flops": 6 * T * D * I}
    return {"bytes": c["E"] * c["D"] * 4 + c["D"] * 4, "flops": 2 * c["E"] * c["D"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "router":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "stack":                           # a rounding of one layer travels through the next
        return {"rel": 1e-5, "max": 4e-4}
    # 32-bit sums; the Inkling layer's shared experts round their activations to bf16, where a
    # last bit of the hidden activations moves a rounding now and then
    if kind == "layer" and case["shared"] == cf.SHARED_GATED:
        return {"rel": 2e-4, "max": 1e-2}
    if kind == "matmul" and case["weights"] == "bf16_rx":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 4e-6, "max": 2e-4}


# ------------------------------------------------------------------ exact ----

def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _expert(gu, dn, e, I, D, x):
    g = _unq4(gu[0][e * 2 * I:(e + 1) * 2 * I], gu[1][e * 2 * I:(e + 1) * 2 * I])
    y = x @ g.T.contiguous()
    h = _silu(y[:, :I]) * y[:, I:]
    return h @ _unq4(dn[0][e * D:(e + 1) * D], dn[1][e * D:(e + 1) * D]).T.contiguous()


def _route(cfg, w, x):
    """(picks, weights, shared gates' weights) in 64 bits"""
    lg = x @ w["router"].double().T.contiguous()
    act, E, K = cfg.route_act, cfg.E, cfg.K
    if act in (cf.ROUTE_SOFTMAX, cf.ROUTE_SOFTMAX_OLMOE, cf.ROUTE_SOFTMAX_QWEN):
        sc = torch.softmax(lg, 1)
    elif act in (cf.ROUTE_SOFTPLUS, cf.ROUTE_SQRT_SOFTPLUS):
        sc = torch.log1p(torch.exp(lg))
        sc = sc.sqrt() if act == cf.ROUTE_SQRT_SOFTPLUS else sc
    else:
        sc = torch.sigmoid(lg)
    key = sc[:, :E] + w["corr_bias"].double() if "corr_bias" in w else sc[:, :E]
    sel = torch.topk(key, K, dim=1).indices
    wt = sc.gather(1, sel)
    if act == cf.ROUTE_INKLING:
        f = cfg.route_scale / (wt.sum(1, keepdim=True) + sc[:, E:].sum(1, keepdim=True))
        return sel, wt * f, sc[:, E:] * f
    if cfg.norm_topk or act == cf.ROUTE_SOFTMAX_QWEN:
        wt = wt / wt.sum(1, keepdim=True)
    return sel, wt * cfg.route_scale, None


def _moe(cfg, w, x):
    sel, wt, wsh = _route(cfg, w, x)
    acc = torch.zeros_like(x)
    for e in range(cfg.E):
        s, k = torch.nonzero(sel == e, as_tuple=True)
        if len(s):
            y = _expert((w["gu_q"], w["gu_s"]), (w["dn_q"], w["dn_s"]), e, cfg.I, cfg.D, x[s])
            acc.index_add_(0, s, y * wt[s, k][:, None])
    bf = lambda v: v.float().to(torch.bfloat16).double()
    for j in range(cfg.n_shared_experts):
        r, d = slice(j * cfg.Is, (j + 1) * cfg.Is), slice(j * cfg.D, (j + 1) * cfg.D)
        gated = cfg.shared_mode == cf.SHARED_GATED            # its matmuls round their activations to bf16
        xx = bf(x) if gated else x
        h = _silu(xx @ w["sg"][r].double().T.contiguous()) * (xx @ w["su"][r].double().T.contiguous())
        y = (bf(h) if gated else h) @ w["sd"][d].double().T.contiguous()
        acc += y * wsh[:, j:j + 1] if gated else y
    return acc


def _rms(h, w):
    return h / torch.sqrt((h * h).mean(1, keepdim=True) + NORM_EPS) * w.double()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "layer":
        cfg, w, x, res = _inputs(c, seed)
        return res.double() + _moe(cfg, w, x.double())
    if kind == "stack":
        cfg, ws, norms, head, x = _inputs(c, seed)
        h = x.double()
        for i, w in enumerate(ws):
            h = h + _moe(cfg, w, _rms(h, norms[i]))
        return {"h": h, "logits": _rms(h, norms[-1]) @ head.double().T.contiguous()}
    if kind == "group":
        gu, dn, x, (sel, wts, *_) = _inputs(c, seed)
        x, sel, wts = (torch.from_numpy(a).cuda() for a in (x, sel, wts))
        acc = torch.zeros(c["S"], c["D"], dtype=torch.float64, device="cuda")
        for e in range(c["E"]):
            s, k = torch.nonzero(sel == e, as_tuple=True)
            if len(s):
                acc.index_add_(0, s, _expert(gu, dn, e, c["I"], c["D"], x[s].double()) * wts[s, k].double()[:, None])
        return acc
    if kind == "matmul":
        W, x = _inputs(c, seed)
        x = torch.from_numpy(x).cuda()
        if c["weights"] == "bf16_rx" and c["I"] % 32 == 0:    # activations rounded to bf16
            x = x.to(torch.bfloat16)
        if c["weights"].startswith("bf16"):
            w = W[0].double()
        elif c["weights"] == "q8":
            w = W[0].double() * W[1].double()[:, None]
        else:
            w = _unq4(*W)
        return x.double() @ w.T.contiguous()
    if kind == "glm":
        ts, x = _inputs(c, seed)
        x = torch.from_numpy(x).cuda().double().view(c["experts"], c["rows"], c["D"])
        out = []
        for e, (g, u, d) in enumerate(ts):
            h = _silu(x[e] @ _unq4(*g).T.contiguous()) * (x[e] @ _unq4(*u).T.contiguous())
            out.append(h @ _unq4(*d).T.contiguous())
        return torch.cat(out)
    W, b, x = _inputs(c, seed)
    sc = torch.sigmoid(W.double() @ x.double())
    sel = torch.topk(sc + b.double(), c["K"]).indices
    return {"idx": None, "w": sc[sel] / sc[sel].sum()}
