"""The measured workloads of the routed VQ expert path.

Each case is a call that a program using this package makes, through the
package's public entry points, at sizes from its own configurations (the
384-expert 4096/2048 top-6 layer, the 288-expert 4096/1536 top-8 layer with the
nested tier, the 4096 -> 2048 projection) and at generic ones. Kinds:

- ``linear``: ``QuantizedVQLinear`` on rows of activations;
- ``moe``: ``RoutedVQMoE`` (router logits -> routed SwiGLU experts -> combine);
- ``switch``: ``QuantizedVQSwitchLinear``, one routed projection;
- ``verify``: ``gather_vqmm_verify_rows`` grouped by expert;
- ``quantize``: ``quantize_weight_rtn`` of a dense weight.

Codes are uniform, as a trained quantiser's are close to; scales are fp16,
log-normal about 0.02; activations are N(0, 1), as they are after the RHT.
"""

from __future__ import annotations

import itertools
import math

import torch

import keep_amd

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}
OFF = -1.0e30  # router bias of an expert that is not resident


def listed():
    return [
        # one token through one dense projection: the smallest call, all latency
        _linear("linear_row", 1, 4096, 2048, bits=16, group=0, dtype="float16"),
        # a prompt through a dense layer in the default format (8-bit E8, groups of 512) with its input RHT
        _linear("linear_prefill", 2048, 4096, 4096, bits=8, group=512, dtype="bfloat16", rht=True),
        # one token through the 384-expert layer: batch-1 decode, the headline
        _moe("moe_decode_1", 1, 384, 6, 4096, 2048, dtype="float16"),
        # a speculative-verify window of 8 tokens through the same layer
        _moe("moe_verify_8", 8, 384, 6, 4096, 2048, dtype="float16"),
        # the largest window of the few-token path, inside a whole block: shared expert, residual, bf16
        _moe("moe_block_64", 64, 384, 6, 4096, 2048, dtype="bfloat16", shared=True),
        # a prompt of 2048 tokens, skewed expert popularity
        _moe("moe_prefill_2048", 2048, 384, 6, 4096, 2048, dtype="float16", routing="zipf"),
        # decode with half of the experts resident and the nested 3-bit tier on 28 of them
        _moe("moe_tier_1", 1, 288, 8, 4096, 1536, dtype="bfloat16", resident=0.5, hot=28),
        # a prompt through that layer
        _moe("moe_tier_prefill_512", 512, 288, 8, 4096, 1536, dtype="bfloat16", resident=0.5, hot=28),
        # a hidden size beyond 4096 with grouped scales, a small decode batch
        _moe("moe_wide_4", 4, 128, 8, 7168, 2048, group=512, dtype="bfloat16"),
        # the verify-rows operator in its 8-bit format, 8 rows, top-6 of 256
        _routed("verify", "verify_8", 8, 256, 6, 4096, 2048, bits=8, group=512, dtype="float16"),
        # a prompt, of an odd length, through one routed projection in the default 8-bit format
        _routed("switch", "switch_prefill_333", 333, 256, 6, 4096, 2048, bits=8, group=512, dtype="bfloat16"),
        # a dense weight quantised to E8P on the device
        {"name": "quantize_e8p", "kind": "quantize", "out_dims": 2048, "in_dims": 4096, "group": 512, "bits": 16},
    ]


def _linear(name, rows, in_dims, out_dims, *, bits, group, dtype, rht=False):
    return {"name": name, "kind": "linear", "rows": rows, "in_dims": in_dims, "out_dims": out_dims, "bits": bits,
            "group": group, "dtype": dtype, "rht": rht}


def _moe(name, tokens, experts, top_k, hidden, inter, *, dtype, group=0, routing="normal", resident=1.0, hot=0,
         shared=False):
    return {"name": name, "kind": "moe", "tokens": tokens, "experts": experts, "top_k": top_k, "hidden": hidden,
            "inter": inter, "group": group, "dtype": dtype, "routing": routing, "resident": resident, "hot": hot,
            "shared": shared}


def _routed(kind, name, tokens, experts, top_k, in_dims, out_dims, *, bits, group, dtype):
    return {"name": name, "kind": kind, "tokens": tokens, "experts": experts, "top_k": top_k, "in_dims": in_dims,
            "out_dims": out_dims, "bits": bits, "group": group, "dtype": dtype}


def _log(rng, lo, hi):
    """A whole number of lo..hi, spread evenly over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["linear", "linear", "moe", "moe", "moe", "tier", "verify", "switch", "quantize"])
    dtype = rng.choice(["float16", "bfloat16"])
    if kind == "linear":
        bits, K = rng.choice([8, 16]), rng.choice([1024, 2048, 4096])
        return _unnamed(_linear("", _log(rng, 1, 2048), K, 8 * rng.randint(64, 512), bits=bits,
                                group=rng.choice([0, 512]), dtype=dtype, rht=rng.random() < 0.5))
    if kind in ("verify", "switch"):
        tokens = _log(rng, 2, 16) if kind == "verify" else _log(rng, 1, 333)
        return _unnamed(_routed(kind, "", tokens, rng.randint(16, 256), rng.randint(2, 6),
                                512 * rng.randint(2, 8), 8 * rng.randint(64, 256), bits=rng.choice([8, 16]), group=512,
                                dtype=dtype))
    if kind == "quantize":
        return {"kind": "quantize", "out_dims": rng.randint(200, 2048), "in_dims": 512 * rng.randint(1, 8),
                "group": rng.choice([128, 512]), "bits": rng.choice([8, 16])}
    if kind == "tier":
        experts = 8 * rng.randint(8, 36)
        return _unnamed(_moe("", rng.choice([1, _log(rng, 32, 512)]), experts, 8, 4096, 512 * rng.randint(1, 3),
                             dtype=dtype, resident=0.5, hot=max(1, experts // 10)))
    hidden, inter = rng.choice([(2048, 768), (2880, 1440), (4096, 1536), (4096, 2048), (5120, 1536), (7168, 2048)])
    ragged = hidden == 2880  # no scale group of 512 and no 128-wide K blocks
    top_k = rng.randint(4, 8)
    tokens = _log(rng, 1, 24 if ragged else min(2048, int(6e11 / (6 * top_k * hidden * inter))))
    group = 0 if ragged or inter % 512 else rng.choice([0, 512])
    return _unnamed(_moe("", tokens, 8 * rng.randint(4, 16 if hidden > 4096 else 48), top_k, hidden, inter,
                         dtype=dtype, group=group, routing=rng.choice(["normal", "zipf"]),
                         shared=rng.random() < 0.3))


def _unnamed(case):
    del case["name"]
    return case


# --------------------------------------------------------------------------- inputs


class _Inputs:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(shape, device=self.dev, generator=self.g, dtype=torch.float32)

    def codes(self, bits, *shape):
        if bits == 8:
            return torch.randint(0, 256, shape, dtype=torch.uint8, device=self.dev, generator=self.g)
        return torch.randint(-32768, 32768, shape, dtype=torch.int16, device=self.dev, generator=self.g)

    def scales(self, *shape):
        return (0.02 * torch.exp(0.3 * self.normal(*shape))).half()

    def signs(self, n):
        return torch.randint(0, 2, (n,), device=self.dev, generator=self.g).float() * 2 - 1

    def perm(self, n):
        return torch.randperm(n, device=self.dev, generator=self.g)


def _make(case, seed):
    """The raw tensors of a case."""
    m, c = _Inputs(seed), case
    d = {}
    if c["kind"] == "quantize":
        return {"weight": 0.02 * m.normal(c["out_dims"], c["in_dims"])}
    dt = _DTYPES[c["dtype"]]
    if c["kind"] == "linear":
        K, N, g = c["in_dims"], c["out_dims"], c["group"] or c["in_dims"]
        d["codes"], d["scales"] = m.codes(c["bits"], N, K // 8), m.scales(N, K // g)
        d["x"] = m.normal(c["rows"], K).to(dt)
        d["signs"] = m.signs(K) if c["rht"] else None
        return d
    E, T, k = c["experts"], c["tokens"], c["top_k"]
    if c["kind"] in ("verify", "switch"):
        K, N, g = c["in_dims"], c["out_dims"], c["group"]
        d["codes"], d["scales"] = m.codes(c["bits"], E, N, K // 8), m.scales(E, N, K // g)
        d["x"] = m.normal(T, K).to(dt)
        d["idx"] = torch.topk(m.normal(T, E), k, dim=-1).indices.to(torch.int32)
        return d
    H, I = c["hidden"], c["inter"]
    for name, n, K in (("gate", I, H), ("up", I, H), ("down", H, I)):
        d[name] = (m.codes(16, E, n, K // 8), m.scales(E, n, K // (c["group"] or K)))
        if c["hot"]:
            d["res_" + name] = (m.codes(8, c["hot"], n, K // 8), (0.1 * m.scales(c["hot"], n, 1).float()).half())
        if c["shared"]:
            d["shared_" + name] = (m.codes(16, 1, n, K // 8), m.scales(1, n, K // (c["group"] or K)))
    d["x"] = m.normal(T, H).to(dt)
    d["residual"] = m.normal(T, H).to(dt) if c["shared"] else None
    z = m.normal(T, E)
    if c["routing"] == "zipf":  # popularity rank^-1.1 under a seeded order, per-token noise on top
        u = torch.rand((T, E), device=m.dev, generator=m.g, dtype=torch.float32).clamp(1e-7, 1 - 1e-7)
        z = z - torch.log(-torch.log(u)) - 1.1 * torch.log(m.perm(E).float() + 1.0)
    d["logits"] = z
    d["resident"] = None
    if c["resident"] < 1:
        order = m.perm(E)
        n = max(k, round(E * c["resident"]))
        d["resident"] = torch.zeros(E, dtype=torch.bool, device=m.dev)
        d["resident"][order[:n]] = True
        if c["hot"]:
            d["hot_rows"] = torch.full((E,), -1, dtype=torch.int32, device=m.dev)
            d["hot_rows"][order[:c["hot"]]] = torch.arange(c["hot"], dtype=torch.int32, device=m.dev)
    return d


def _glu(d, prefix, E, H, I, group, tier=None):
    def lin(name, K, N):
        codes, scales = d[prefix + name]
        return keep_amd.QuantizedVQSwitchLinear(input_dims=K, output_dims=N, num_experts=E, codes=codes,
                                                scales=scales, group_size=group or K, code_bits=16)

    return keep_amd.QuantizedVQSwitchGLU(gate_proj=lin("gate", H, I), up_proj=lin("up", H, I),
                                         down_proj=lin("down", I, H), hot_tier=tier)


def prepare(case, seed):
    c, d = case, _make(case, seed)
    if c["kind"] == "quantize":
        return dict(case=c, weight=d["weight"])
    s = dict(case=c, x=d["x"])
    if c["kind"] == "linear":
        s["layer"] = keep_amd.QuantizedVQLinear(input_dims=c["in_dims"], output_dims=c["out_dims"], codes=d["codes"],
                                                scales=d["scales"], group_size=c["group"] or c["in_dims"],
                                                code_bits=c["bits"], rht_signs=d["signs"])
    elif c["kind"] == "switch":
        s["layer"] = keep_amd.QuantizedVQSwitchLinear(input_dims=c["in_dims"], output_dims=c["out_dims"],
                                                      num_experts=c["experts"], codes=d["codes"],
                                                      scales=d["scales"], group_size=c["group"], code_bits=c["bits"])
        s["idx"] = d["idx"]
    elif c["kind"] == "verify":
        s.update(codes=d["codes"], scales=d["scales"], idx=d["idx"])
    else:
        E, H, I, g = c["experts"], c["hidden"], c["inter"], c["group"]
        tier = None
        if c["hot"]:
            tier = keep_amd.HotTier(d["hot_rows"], {n: d["res_" + n] for n in ("gate", "up", "down")})
        bias = None if d["resident"] is None else keep_amd.resident_bias(d["resident"])
        shared = _glu(d, "shared_", 1, H, I, g) if c["shared"] else None
        s["layer"] = keep_amd.RoutedVQMoE(_glu(d, "", E, H, I, g, tier), top_k=c["top_k"], bias_served=bias,
                                          tau=0.3 if bias is not None else float("inf"), shared_experts=shared,
                                          out_dtype=_DTYPES[c["dtype"]] if c["shared"] else torch.float32)
        s.update(logits=d["logits"], residual=d["residual"])
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "quantize":
        q = keep_amd.quantize_weight_rtn(s["weight"], group_size=c["group"], code_bits=c["bits"])
        return {"codes": q.codes, "scales": q.scales}
    if c["kind"] == "linear":
        return s["layer"](s["x"])
    if c["kind"] == "switch":
        return s["layer"](s["x"], s["idx"])
    if c["kind"] == "verify":
        return keep_amd.gather_vqmm_verify_rows(s["x"], s["codes"], s["scales"], None, s["idx"],
                                                input_dims=c["in_dims"], output_dims=c["out_dims"],
                                                group_size=c["group"], grouping="expert")
    out, r = s["layer"](s["x"], s["logits"], residual=s["residual"])
    return {"out": out, "idx": r.idx, "weight": r.weight, "want": r.want, "want_score": r.want_score,
            "admit": r.admit}


# --------------------------------------------------------------------------- work and tolerance


def _hit(pool, routes, top_k):
    """Experts of a pool that are hit by `routes` routes, on average, popularity aside."""
    tokens = routes / top_k
    return pool * (1.0 - (1.0 - min(1.0, top_k / pool)) ** tokens)


def work(case):
    c = case
    if c["kind"] == "quantize":
        n = c["out_dims"] * c["in_dims"]
        # the factored search: two shifts, 256 rows, eight terms of a subtraction, a product and a sum
        return {"bytes": 4.0 * n + n / 8 * c["bits"] / 8 + 2 * n / c["group"],
                "flops": (n / 8) * (2 if c["bits"] == 16 else 1) * 256 * 24.0}
    if c["kind"] == "linear":
        M, K, N = c["rows"], c["in_dims"], c["out_dims"]
        return {"bytes": N * K / 8 * c["bits"] / 8 + 2 * N * K / (c["group"] or K) + 2 * M * (K + N),
                "flops": 2.0 * M * K * N}
    T, k = c["tokens"], c["top_k"]
    R = T * k
    if c["kind"] in ("verify", "switch"):
        K, N = c["in_dims"], c["out_dims"]
        hit = _hit(c["experts"], R, k)
        return {"bytes": hit * (N * K / 8 * c["bits"] / 8 + 2 * N * K / c["group"]) + 2 * T * K + 4 * R + 2 * R * N,
                "flops": 2.0 * R * K * N}
    H, I = c["hidden"], c["inter"]
    pool = max(k, round(c["experts"] * c["resident"]))
    hit = _hit(pool, R, k)
    group = c["group"]
    expert = 3 * H * I / 4 + 2 * (2 * I * (H // (group or H)) + H * (I // (group or I)))
    tier = 3 * H * I / 8 + 2 * (2 * I + H)
    nbytes = hit * expert + _hit(pool, R, k) * c["hot"] / pool * tier
    flops = 6.0 * R * H * I * (1 + c["hot"] / pool)
    out = 4 * T * H
    if c["shared"]:
        nbytes += expert + 2 * T * H
        flops += 6.0 * T * H * I
        out = 2 * T * H
    return {"bytes": nbytes + 2 * T * H + 4 * T * c["experts"] + out + 17 * R, "flops": flops}


def tolerance(case):
    """About four times the distance seen from the 64-bit result, rounding of the outputs included: 2.1e-4 for
    fp16 outputs, 1.6e-3 for bf16, 2.3e-3 where the RHT's output is rounded to bf16 too, 1.7e-3 to 2.2e-3 for the
    MoE layer (its SwiGLU output is held in bf16)."""
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "moe":
        return {"rel": 8e-3, "differ": 1e-3}
    if case["dtype"] == "float16":
        return {"rel": 1e-3}
    return {"rel": 9e-3 if case.get("rht") else 7e-3}


# --------------------------------------------------------------------------- the same in 64 bits

_PAD = ("31113333 13113333 11313333 11133333 33313311 33313131 33311331 33313113 33311313 33311133 33133311 33133131 "
        "33131331 33133113 33131313 33131133 31333311 31333131 31331331 31333113 31331313 13331133 13333311 13333131 "
        "13331331 13333113 13331313 11331333 33113331").split()


def _e8p_values(dev):
    """Every E8P codeword's eight values, float64 [65536, 8], from the format's definition."""
    low = [r for r in itertools.product((1, 3, 5, 7), repeat=8) if sum(v * v for v in r) <= 40]
    rows = torch.tensor(low + [tuple(int(v) for v in p) for p in _PAD], dtype=torch.int64)
    nib = rows[:, [0, 2, 4, 6, 1, 3, 5, 7]].clone()  # packed order
    odd = nib.sum(1) % 4 == 2
    nib[odd, 7] = -nib[odd, 7]
    code = torch.arange(65536)
    sign, row = code & 255, code >> 8
    parity = torch.zeros_like(sign)
    for b in range(8):
        parity ^= (sign >> b) & 1
    eff = sign ^ parity
    out = torch.empty((65536, 8), dtype=torch.float64)
    for d, n in enumerate((0, 4, 1, 5, 2, 6, 3, 7)):
        v = nib[row, n].double() * 0.5
        out[:, d] = torch.where((eff >> n) & 1 == 1, -v, v) + 0.25 - 0.5 * parity.double()
    return out.to(dev)


def _e8_values(dev):
    """Every 8-bit E8 code's eight values, float64 [256, 8]."""
    ints = [tuple(2 * v for v in r) for r in itertools.product((-1, 0, 1), repeat=8)
            if sum(v * v for v in r) <= 2 and sum(r) % 2 == 0]
    halves = [r for r in itertools.product((-1, 1), repeat=8) if sum(r) % 4 == 0]
    pads = [tuple(s * 4 * (a == d) for d in range(8)) for s in (1, -1) for a in range(8)][:15]
    return (torch.tensor(ints + halves + pads, dtype=torch.float64) * 0.5).to(dev)


def _dense(values, codes, scales):
    """float64 [N, K] of one matrix's codes and scales."""
    W = values[codes.long() & (values.shape[0] - 1)]  # [N, K/8, 8]
    N, G = scales.shape
    return (W.reshape(N, G, -1) * scales.double()[:, :, None]).reshape(N, -1)


def _hadamard(n, dev):
    h = torch.ones((1, 1), dtype=torch.float64, device=dev)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(n)


def exact(case, seed):
    c, d = case, _make(case, seed)
    if c["kind"] == "quantize":
        g = d["weight"].double().abs().reshape(c["out_dims"], -1, c["group"]).amax(-1)
        top = 2.75 if c["bits"] == 16 else 2.0  # the codebooks' largest magnitudes
        return {"codes": None, "scales": g / top}
    x = d["x"].double()
    dev = x.device
    if c["kind"] != "moe":
        values = _e8p_values(dev) if c["bits"] == 16 else _e8_values(dev)
    if c["kind"] == "linear":
        if d["signs"] is not None:
            x = (x * d["signs"].double()) @ _hadamard(c["in_dims"], dev)
        return x @ _dense(values, d["codes"], d["scales"]).t().contiguous()
    T, k = c["tokens"], c["top_k"]
    if c["kind"] in ("verify", "switch"):
        out = torch.empty((T, k, c["out_dims"]), dtype=torch.float64, device=dev)
        for e in d["idx"].unique().tolist():
            t, j = torch.nonzero(d["idx"] == e, as_tuple=True)
            out[t, j] = x[t] @ _dense(values, d["codes"][e], d["scales"][e]).t().contiguous()
        return out
    p = torch.softmax(d["logits"].double(), -1)
    key = p if d["resident"] is None else torch.where(d["resident"], p, torch.full_like(p, OFF))
    idx = torch.topk(key, k, dim=-1).indices
    w = p.gather(-1, idx)
    w = w / w.sum(-1, keepdim=True)
    want = torch.topk(p, k, dim=-1).indices
    base, res = _e8p_values(dev), _e8_values(dev)

    def swiglu(rows, prefix, e, hot):
        def proj(v, name):
            W = _dense(base, d[prefix + name][0][e], d[prefix + name][1][e])
            if hot >= 0:
                W = W + _dense(res, d["res_" + name][0][hot], d["res_" + name][1][hot])
            return v @ W.t().contiguous()
        return proj(torch.nn.functional.silu(proj(rows, "gate")) * proj(rows, "up"), "down")

    out = torch.zeros((T, c["hidden"]), dtype=torch.float64, device=dev)
    hot = d["hot_rows"].tolist() if c["hot"] else None
    for e in idx.unique().tolist():
        t, j = torch.nonzero(idx == e, as_tuple=True)
        out.index_add_(0, t, w[t, j, None] * swiglu(x[t], "", e, hot[e] if hot else -1))
    if c["shared"]:
        out = d["residual"].double() + out + swiglu(x, "shared_", 0, -1)
    return {"out": out, "idx": idx.to(torch.int32), "weight": w, "want": want.to(torch.int32),
            "want_score": p.gather(-1, want), "admit": None}
