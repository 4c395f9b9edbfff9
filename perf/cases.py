"""What the framework's speed is measured on: the work its callers have it do on the GPU.

A case is one call of a public entry point (or the few calls that make one decode step), at the shapes of
this repository's own configurations: hidden 2048, 64 / 128 / 256 experts, 6 to 10 used per token,
intermediate 256 / 512 / 768, Q4_K up and gate, Q4_K or Q6_K down, an always-on shared expert or none.  Four kinds:

  token   MoeCache.decode_token: one token over every layer of a cache (ids back, observed, stepped)
  chain   MoeCache.decode_layer per layer, each layer's input made from the layer below, then observe and step
  batch   MoeCache.decode_batch: several sequences, or a whole prompt chunk, over every layer
  layer   BatchedMoe.forward: one layer over a batch with the caller's own buffers (route, dispatch, experts)

Weights are random Q4_K / Q6_K blocks whose values are about N(0, 0.02), activations N(0, 1), routers
N(0, 0.02) (so logits of standard deviation 0.9 and mildly uneven expert loads), given logits uniform on
[0, 1).  The layers of one cache share their expert bytes (each layer has its own copy in its slots and
its own router), so that a deep cache is quick to make.

Every output is defined to the last bit: integer dots of the quantized values, fp32 only where ggml has
it and in its order, a canonical order for the router and the combine.  So the tolerance is "exact" for
floats too; exact() gives the same chain, with its Q8_K activation codes, in 64 bits.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "moe-prefetch_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from moe_prefetch import MoeCache, TYPE_Q4K, TYPE_Q6K, lib  # noqa: E402
from moe_prefetch.batched import BatchedMoe  # noqa: E402

H = 2048
QK = 256
SIGMA = 0.02
RESIDUAL = 0.25         # a chain's x_{l+1} = x_l + RESIDUAL * out_l stays near unit size without a norm
DEV = "cuda:0"


# ---- the cases ----------------------------------------------------------------
def _case(kind, layers=1, tokens=1, E=128, K=8, I=768, down="q4", shared=False, resident=None, dtype="f32",
          router=True, name=None):
    """down: q4, q6 or alt (Q6_K in odd layers); resident: experts of each layer in HBM slots (the others are read
    from the pinned store); dtype: of a layer case's activations; router: logits from W . x, else given."""
    c = dict(kind=kind, layers=layers, tokens=tokens, E=E, K=K, I=I, down=down, shared=shared,
             resident=E if resident is None else resident, dtype=dtype, router=router)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # batch-1 decode of a model whose one MoE layer sits in HBM: the smallest call, all latency
        _case("token", name="token_1_layer"),
        # batch-1 decode over a whole 48-layer model, Q6_K down in every other layer: the flagship workload's GPU side
        _case("token", layers=48, down="alt", name="token_48_layers"),
        # batch-1 decode through the per-layer op, as a model's graph calls it: 256 experts and a shared one
        _case("chain", layers=8, E=256, I=512, shared=True, name="chain_8_layers_shared"),
        # batch-1 decode with one expert in eight outside the slots, read from pinned host memory over PCIe
        _case("token", layers=4, resident=112, name="token_4_layers_absent"),
        # a small decode batch of the wide model with its shared expert
        _case("batch", layers=8, tokens=16, E=256, I=512, shared=True, name="batch_16_shared"),
        # a full decode batch: four pairs per expert on average
        _case("batch", layers=8, tokens=64, down="alt", name="batch_64"),
        # a short ragged prompt through a small model's layer
        _case("layer", tokens=37, E=64, K=6, I=256, down="q6", name="layer_37_small"),
        # a ragged prompt chunk of ordinary size
        _case("layer", tokens=197, name="layer_197"),
        # the usual prefill chunk, bf16 activations, logits from the caller's own router
        _case("layer", tokens=512, dtype="bf16", router=False, name="layer_512_bf16"),
        # a longer ragged chunk through the wide model's layer
        _case("layer", tokens=1000, E=256, I=512, down="q6", name="layer_1000_wide"),
        # a long prefill chunk, bf16, Q6_K down
        _case("layer", tokens=2048, down="q6", dtype="bf16", router=False, name="layer_2048_bf16"),
        # the largest chunk the cached path takes in one call
        _case("batch", tokens=4096, name="batch_4096"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("token", "chain", "batch", "layer", "layer", "layer"))
    E = rng.choice((64, 128, 256))
    I = rng.choice((256, 512, 768))
    K = rng.choice((6, 8, 8, 8, 10))
    shared = kind != "layer" and rng.random() < 0.3
    if kind == "token":
        layers = _log_int(rng, 1, 40)
        absent = rng.random() < 0.25 and layers <= 6
        return _case("token", layers, 1, E, K, I, rng.choice(("q4", "q6", "alt")), shared,
                     E - E // 8 if absent else E)
    if kind == "chain":
        return _case("chain", _log_int(rng, 1, 16), 1, E, K, I, rng.choice(("q4", "q6", "alt")), shared)
    if kind == "batch":
        tokens = _log_int(rng, 2, 2500)
        return _case("batch", rng.randint(1, 6) if tokens <= 96 else 1, tokens, E, K if tokens < 2000 else 8, I,
                     rng.choice(("q4", "q6", "alt")), shared and tokens < 1500)
    tokens = _log_int(rng, 1, 3000)
    return _case("layer", 1, tokens, E, K if tokens < 2000 else 8, I, rng.choice(("q4", "q6")),
                 dtype=rng.choice(("f32", "bf16")), router=rng.random() < 0.5)


def _down_type(case, layer):
    return TYPE_Q6K if case["down"] == "q6" or (case["down"] == "alt" and layer % 2) else TYPE_Q4K


def _expert_bytes(I, dt):
    return 2 * I * (H // QK) * 144 + H * (I // QK) * (210 if dt == TYPE_Q6K else 144)


def work(case):
    """Each expert that some token uses is read once (as many as a uniform routing uses on average), the router and
    the activations once, and the outputs written; a multiply-add per weight and pair is two operations."""
    T, K, E, I, NL = case["tokens"], case["K"], case["E"], case["I"], case["layers"]
    used = E * (1.0 - (1.0 - K / E) ** T)
    b = f = 0.0
    for l in range(NL):
        b += (used + bool(case["shared"])) * _expert_bytes(I, _down_type(case, l))
        b += T * H * ((2 if case["dtype"] == "bf16" else 4) + 4) + T * K * 8
        f += 2.0 * T * (K + bool(case["shared"])) * 3 * H * I
        if case["router"]:
            b += 4.0 * E * H
            f += 2.0 * T * E * H
        else:
            b += 4.0 * T * E
    return {"bytes": b, "flops": f}


def tolerance(case):
    return "exact"


# ---- inputs -------------------------------------------------------------------
def _gen(seed, what):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + what * 7919 + 12345) % (1 << 62))
    return g


def _fp16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _q4k_blocks(n, g):
    """n Q4_K blocks [n][144]: fp16 d and dmin, eight six-bit (scale, min) pairs, 256 nibbles; values about N(0, SIGMA)."""
    d = SIGMA * 0.33 / 52 * (0.9 + 0.2 * torch.rand(n, device=DEV, generator=g))
    sc = torch.randint(40, 64, (n, 8), device=DEV, generator=g)
    mn = torch.randint(40, 64, (n, 8), device=DEV, generator=g)
    q = torch.randn((n, 256), device=DEV, generator=g).mul_(3.0).add_(7.5).round_().clamp_(0, 15).to(torch.uint8)
    s = torch.empty((n, 12), dtype=torch.int64, device=DEV)
    s[:, 0:4] = sc[:, :4] | (sc[:, 4:] >> 4 << 6)
    s[:, 4:8] = mn[:, :4] | (mn[:, 4:] >> 4 << 6)
    s[:, 8:12] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    q = q.view(n, 4, 2, 32)
    return torch.cat([_fp16_bytes(d), _fp16_bytes(7.5 * d), s.to(torch.uint8), (q[:, :, 0] | q[:, :, 1] << 4).view(n, 128)], 1)


def _q6k_blocks(n, g):
    """n Q6_K blocks [n][210]: 256 six-bit values (low nibbles, then high pairs), 16 int8 scales, fp16 d."""
    d = SIGMA / 10.0 / 90 * (0.9 + 0.2 * torch.rand(n, device=DEV, generator=g))
    sc = torch.randint(60, 121, (n, 16), device=DEV, generator=g)
    sc = torch.where(torch.rand((n, 16), device=DEV, generator=g) < 0.5, -sc, sc).to(torch.int8)
    q = torch.randn((n, 256), device=DEV, generator=g).mul_(10.0).add_(32.0).round_().clamp_(0, 63).to(torch.uint8)
    q = q.view(n, 2, 4, 32)
    lo, hi = q & 15, q >> 4
    ql = torch.cat([lo[:, :, 0] | lo[:, :, 2] << 4, lo[:, :, 1] | lo[:, :, 3] << 4], 2).view(n, 128)
    qh = (hi[:, :, 0] | hi[:, :, 1] << 2 | hi[:, :, 2] << 4 | hi[:, :, 3] << 6).view(n, 64)
    return torch.cat([ql, qh, sc.view(torch.uint8), _fp16_bytes(d)], 1)


def _experts(n, I, dt, seed, what):
    """[n][expert bytes] in HBM: up, gate (Q4_K rows of H values), down (rows of I values)."""
    g = _gen(seed, what)
    out = torch.empty((n, _expert_bytes(I, dt)), dtype=torch.uint8, device=DEV)
    gu, dn = 2 * I * (H // QK), H * (I // QK)
    for e in range(0, n, 16):
        m = min(16, n - e)
        out[e:e + m, :gu * 144] = _q4k_blocks(m * gu, g).view(m, -1)
        out[e:e + m, gu * 144:] = (_q6k_blocks if dt == TYPE_Q6K else _q4k_blocks)(m * dn, g).view(m, -1)
    return out


def _types(case):
    return sorted({_down_type(case, l) for l in range(case["layers"])})


def _store_of(case, seed, dt):
    return _experts(case["E"], case["I"], dt, seed, dt)


def _shared_of(case, seed, dt):
    return _experts(1, case["I"], dt, seed, 50 + dt) if case["shared"] else None


def _vectors(case, seed):
    """router weights [L][E][H] (or None), given logits [T][E] (or None), activations [L][T][H] f32"""
    NL, T, E = case["layers"], case["tokens"], case["E"]
    W = lg = None
    if case["router"]:
        W = torch.randn((NL, E, H), device=DEV, generator=_gen(seed, 1)).mul_(SIGMA)
    else:
        lg = torch.rand((T, E), device=DEV, generator=_gen(seed, 2))
    n_x = 1 if case["kind"] == "chain" else NL
    x = torch.randn((n_x, T, H), device=DEV, generator=_gen(seed, 3))
    return W, lg, x


class _Cached:
    """A MoeCache over pinned stores, the first `resident` experts of every layer in slots."""

    def __init__(self, case, seed):
        NL, E, K, I = case["layers"], case["E"], case["K"], case["I"]
        self.host = {}
        L = lib()
        for dt in _types(case):
            b = _store_of(case, seed, dt)
            p = L.moe_host_alloc(b.numel())
            if not p:
                raise MemoryError("out of memory: pinned store of %d bytes" % b.numel())
            self.host[dt] = p
            torch.from_numpy(np.ctypeslib.as_array((ctypes.c_uint8 * b.numel()).from_address(p))).copy_(b.view(-1))
            del b
        self.W, _, self.x = _vectors(case, seed)
        res = case["resident"]
        self.cache = c = MoeCache(NL, n_experts=E, n_expert_used=K, intermediate=I, n_slots=res, max_inserts=res,
                                  down_types=[_down_type(case, l) for l in range(NL)], batch_tables=True, device=0)
        shared = {dt: _shared_of(case, seed, dt) for dt in _types(case)}
        warm = np.arange(res, dtype=np.int32)
        for l in range(NL):
            dt = _down_type(case, l)
            c.set_host_store(l, self.host[dt])
            c.set_router(l, self.W[l])
            if shared[dt] is not None:
                c.set_shared(l, shared[dt])
            c.observe(l, warm, n_tok=res)
        c.step()                # schedules the uploads of the experts observed
        c.sync()
        c.step()                # publishes them
        for l in range(NL):
            assert (c.table(l)[0] < res).sum() == res
        if res < E:
            c.freeze()          # which experts are absent stays the same from pass to pass

    def __del__(self):
        if sys is None or sys.is_finalizing():
            return
        torch.cuda.synchronize()
        self.cache.close()
        for p in self.host.values():
            lib().moe_host_free(p)


def prepare(case, seed):
    NL, T, E, K, I = (case[k] for k in ("layers", "tokens", "E", "K", "I"))
    s = {"case": case, "stream": torch.cuda.current_stream().cuda_stream}
    if case["kind"] == "layer":
        dt = _down_type(case, 0)
        s["store"] = _store_of(case, seed, dt)
        W, s["logits"], x = _vectors(case, seed)
        s["W"] = None if W is None else W[0]
        s["xf"] = x[0]
        s["x"] = x[0].to(torch.bfloat16) if case["dtype"] == "bf16" else x[0]
        s["moe"] = BatchedMoe(T, n_experts=E, n_expert_used=K, intermediate=I)
        s["out"] = torch.empty((T, H), device=DEV)
        s["dt"], s["eb"] = dt, _expert_bytes(I, dt)
        return s
    s["held"] = h = _Cached(case, seed)
    if case["kind"] == "batch":
        s["x"], s["out"] = h.x, torch.empty((NL, T, H), device=DEV)
        s["ids"] = np.empty((NL, T, K), np.int32)
    elif case["kind"] == "token":
        s["x"], s["out"] = h.x[:, 0].contiguous(), torch.empty((NL, H), device=DEV)
        s["ids"] = np.empty((NL, K), np.int32)
    else:
        s["x"] = h.x[0, 0].contiguous()
        s["out"] = torch.empty((NL, H), device=DEV)
        s["ids"] = torch.empty((NL, K), dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    return s


# ---- one pass -----------------------------------------------------------------
def run(s):
    case, st = s["case"], s["stream"]
    if case["kind"] == "layer":
        m, T = s["moe"], case["tokens"]
        m.forward(s["x"], s["out"], s["store"], s["eb"], case["E"], s["dt"], logits=s["logits"], W=s["W"],
                  xf32=s["xf"], stream=st)
        return {"out": s["out"], "ids": m.ids[:T], "w": m.w[:T]}
    c = s["held"].cache
    if case["kind"] == "token":
        ids = c.decode_token(s["x"], s["out"], stream=st, ids_out=s["ids"])
        return {"out": s["out"], "ids": ids}
    if case["kind"] == "batch":
        ids = c.decode_batch(s["x"], s["out"], stream=st, ids_out=s["ids"])
        return {"out": s["out"], "ids": ids}
    x, out, ids = s["x"], s["out"], s["ids"]
    for l in range(case["layers"]):
        c.decode_layer(l, x, out[l], ids=ids[l], stream=st)
        x = torch.add(x, out[l], alpha=RESIDUAL)
    host = ids.cpu().numpy()
    for l in range(case["layers"]):
        c.observe(l, host[l])
    c.step()
    return {"out": out, "x": x, "ids": host}


# ---- the same in 64 bits --------------------------------------------------------
def _f16_of(b):
    return b.contiguous().view(torch.float16).double()


def _q4k_values(b, rows, n):
    b = b.view(-1, 144)
    d, dm = _f16_of(b[:, 0:2]), _f16_of(b[:, 2:4])
    s = b[:, 4:16].to(torch.int64)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
    q = b[:, 16:].view(-1, 4, 32)
    q = torch.stack([q & 15, q >> 4], 2).view(-1, 8, 32).double()
    return ((d * sc).unsqueeze(2) * q - (dm * mn).unsqueeze(2)).view(rows, n)


def _q6k_values(b, rows, n):
    b = b.view(-1, 210)
    ql, qh = b[:, :128].view(-1, 2, 64), b[:, 128:192].view(-1, 2, 32)
    a, c = ql[:, :, :32], ql[:, :, 32:]
    q = torch.stack([(a & 15) | (qh & 3) << 4, (c & 15) | (qh >> 2 & 3) << 4, (a >> 4) | (qh >> 4 & 3) << 4,
                     (c >> 4) | (qh >> 6) << 4], 2).view(-1, 16, 16).double() - 32.0
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return (_f16_of(b[:, 208:210]).unsqueeze(2) * sc.unsqueeze(2) * q).view(rows, n)


def _q8k(x):
    """x as its Q8_K codes times their block scale: the value of largest magnitude of each 256 becomes -127 steps.  The
    codes are whole numbers that the format takes in fp32 (a bf16 activation often lies halfway between two of them)."""
    v = x.to(torch.float32).reshape(-1, QK)
    mx = v.gather(1, v.abs().argmax(1, keepdim=True))
    s = torch.where(mx == 0, torch.zeros_like(mx), torch.full_like(mx, -127.0) / mx)
    q = (s * v).round().clamp(max=127).double()
    return torch.where(mx == 0, torch.zeros_like(q), q / torch.where(s == 0, torch.ones_like(s), s).double()).reshape(x.shape)


def _expert64(b, I, dt, xq):
    gu = 2 * I * (H // QK) * 144
    w = _q4k_values(b[:gu], 2 * I, H)
    y = xq @ w.t()
    up, gate = y[:, :I], y[:, I:]
    h = _q8k(gate / (1.0 + torch.exp(-gate)) * up)
    return h @ (_q6k_values if dt == TYPE_Q6K else _q4k_values)(b[gu:], H, I).t()


def _layer64(x, logits, store, shared, case, dt):
    """x [T][H], logits [T][E] in 64 bits -> out [T][H], ids, weights"""
    T, E, K, I = x.shape[0], case["E"], case["K"], case["I"]
    p, ids = torch.sort(torch.softmax(logits, 1), dim=1, descending=True, stable=True)
    ids, w = ids[:, :K], p[:, :K] / p[:, :K].sum(1, keepdim=True)
    xq = _q8k(x)
    out = torch.zeros((T, H), dtype=torch.float64, device=DEV)
    for e in ids.unique().tolist():
        t, k = (ids == e).nonzero(as_tuple=True)
        out.index_add_(0, t, _expert64(store[e], I, dt, xq[t]) * w[t, k].unsqueeze(1))
    if shared is not None:
        out += _expert64(shared[0], I, dt, xq)
    return out, ids.to(torch.int32), w


def exact(case, seed):
    W, lg, xs = _vectors(case, seed)
    stores = {dt: _store_of(case, seed, dt) for dt in _types(case)}
    shared = {dt: _shared_of(case, seed, dt) for dt in _types(case)}
    outs, ids, w = [], [], None
    chain = case["kind"] == "chain"
    x = xs[0].double()
    for l in range(case["layers"]):
        dt = _down_type(case, l)
        xr = x if chain else xs[l].double()
        logits = lg.double() if W is None else xr @ W[l].double().t()
        xl = xs[l].to(torch.bfloat16).double() if case["dtype"] == "bf16" else xr
        o, i, w = _layer64(xl, logits, stores[dt], shared[dt], case, dt)
        outs.append(o)
        ids.append(i)
        x = x + RESIDUAL * o
    if case["kind"] == "layer":
        return {"out": outs[0], "ids": ids[0], "w": w}
    if case["kind"] == "batch":
        return {"out": torch.stack(outs), "ids": torch.stack(ids)}
    r = {"out": torch.cat(outs), "ids": torch.cat(ids)}
    return {**r, "x": x[0]} if chain else r
