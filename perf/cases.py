"""The calls that a user of the layer makes, as measurable cases.

Four kinds of call, each through the binding a program uses:

* ``layer``: k3x_hip_moe_forward, the routed-expert layer with device routing (the main path);
* ``official``: k3x_hip_official_prepare + k3x_hip_official_ffn, one step of the official K3 FFN;
* ``latent``: k3x_hip_resident_moe_layer, the fp32 latent layer with routes from the host;
* ``miss``: experts admitted to their slots from device extents (checked against their CRC32C),
  then one token through them with k3x_hip_moe_forward_routed, as a cache of experts does on a miss.

``prepare`` draws inputs and weights from the seed with torch and uploads them; ``exact`` draws the
same ones again and computes the call in float64 with plain torch.  Rounding points that the layer
documents (bf16 of the normalised input and of the GLU output; the official layer's bf16 latent,
expert outputs, mix, gate, up and down) are kept in ``exact``; sums and everything else are 64-bit
and the final outputs are not rounded.
"""
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "project-k3x_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

DEV = "cuda:0"

# The K3-shaped layer and the official layer of the benchmark.
K3 = dict(hidden=7168, inter=2048, experts=384, top_k=16, shared_inter=2048, routed_scale=2.5)
OFFICIAL = dict(hidden=7168, latent=3584, inter=3072, experts=896, top_k=16, shared_inter=6144)
EPS = 1e-6
OFFICIAL_EPS = 1e-5
BETA, LINEAR = 4.0, 25.0
SCALE_LO, SCALE_HI = 119, 123


def listed():
    layer = dict(kind="layer", glu="swiglu", renorm="float", zipf=False, **K3)
    official = dict(kind="official", **OFFICIAL)
    return [
        # The smallest call: one token of a toy layer; launches and latency are all of it.
        dict(layer, name="tiny_t1", tokens=1, hidden=256, inter=512, experts=16, top_k=4,
             shared_inter=0, routed_scale=1.0),
        # Decode, two positions a step: the benchmark's headline call.
        dict(layer, name="decode_t2", tokens=2),
        # A batch of decoding users, odd count, the SiTU activation and double renormalisation.
        dict(layer, name="batch_t13", tokens=13, glu="situ", renorm="double"),
        # Verification window with a skewed router: busy experts serve many of its tokens.
        dict(layer, name="verify_t64", tokens=64, zipf=True),
        # A batch between the window and the chunk kernels.
        dict(layer, name="batch_t97", tokens=97),
        # The ragged last chunk of a prompt.
        dict(layer, name="chunk_t331", tokens=331),
        # A whole prefill chunk.
        dict(layer, name="prefill_t2048", tokens=2048),
        # The official layer: decode, a window or batch, a prefill chunk.
        dict(official, name="official_t2", tokens=2),
        dict(official, name="official_t45", tokens=45),
        dict(official, name="official_t2048", tokens=2048),
        # The fp32 latent layer at the released dimensions, one token, 16 resident experts.
        dict(kind="latent", name="latent_t1", tokens=1, hidden=7168, latent=3584, inter=3072,
             experts=16, top_k=16, shared_inter=6144),
        # A decode token whose routes miss: four official-shape experts admitted, then run.
        dict(kind="miss", name="miss_4", tokens=1, hidden=3584, inter=3072, experts=8, top_k=4),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    u = rng.random()
    if u < 0.45:  # the K3 layer at any token count
        zipf = rng.random() < 0.25
        return dict(kind="layer", glu=rng.choice(["swiglu", "situ"]),
                    renorm=rng.choice(["float", "double"]), zipf=zipf,
                    tokens=_log_int(rng, 1, 2048), **K3)
    if u < 0.7:  # a layer of another shape
        experts = _log_int(rng, 4, 384)
        return dict(kind="layer", glu=rng.choice(["swiglu", "situ"]),
                    renorm=rng.choice(["float", "double"]), zipf=False,
                    tokens=_log_int(rng, 1, 2048), hidden=128 * _log_int(rng, 2, 56),
                    inter=128 * _log_int(rng, 1, 24), experts=experts,
                    top_k=rng.randint(1, min(16, experts)),
                    shared_inter=rng.choice([0, 128 * _log_int(rng, 1, 16)]),
                    routed_scale=rng.choice([1.0, 2.5]))
    if u < 0.85:
        return dict(kind="official", tokens=_log_int(rng, 1, 2048), **OFFICIAL)
    if u < 0.93:
        experts = rng.randint(8, 32)
        return dict(kind="latent", tokens=rng.randint(1, 8), hidden=7168, latent=3584, inter=3072,
                    experts=experts, top_k=rng.randint(1, min(16, experts)), shared_inter=6144)
    return dict(kind="miss", tokens=1, hidden=3584, inter=3072, experts=8, top_k=rng.randint(1, 8))


# ---- inputs from the seed ---------------------------------------------------------------------

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + stream) % (1 << 62))
    return g


def _normal(seed, stream, shape, sigma, dtype=torch.float32):
    t = torch.randn(shape, device=DEV, generator=_gen(seed, stream)) * sigma
    return t.to(dtype)


def _expert(seed, e, hidden, inter):
    """MXFP4 codes [3][n / 2] and scale bytes [3][n / 32] of one expert (gate, up, down)."""
    n = hidden * inter
    g = _gen(seed, 1000 + e)
    codes = torch.randint(0, 256, (3, n // 2), dtype=torch.uint8, device=DEV, generator=g)
    scales = torch.randint(SCALE_LO, SCALE_HI + 1, (3, n // 32), dtype=torch.uint8, device=DEV,
                           generator=g)
    return codes, scales


def _extents(codes, scales):
    return [codes[0], scales[0], codes[1], scales[1], codes[2], scales[2]]


def _router(seed, c, dtype=torch.float32):
    """Router rows ~ N(0, 0.02^2), correction bias ~ N(0, 0.1^2) or Zipf over shuffled experts."""
    w = _normal(seed, 1, (c["experts"], c["hidden"]), 0.02, dtype)
    if c.get("zipf"):
        order = torch.randperm(c["experts"], device=DEV, generator=_gen(seed, 2))
        rank = torch.argsort(order) + 1
        bias = (0.45 * rank.double() ** -1.1).float()
    else:
        bias = _normal(seed, 2, (c["experts"],), 0.1)
    return w, bias


def _shared(seed, c, hidden, sigma=0.02, dtype=torch.bfloat16):
    s = c["shared_inter"]
    return [_normal(seed, 3 + i, shape, sigma, dtype)
            for i, shape in enumerate([(s, hidden), (s, hidden), (hidden, s)])]


def _host_bits(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


def _official_weights(seed, c):
    h, lat = c["hidden"], c["latent"]
    b = torch.bfloat16
    w = dict(routed_down=_normal(seed, 10, (lat, h), 0.02, b),
             routed_norm=_normal(seed, 11, (lat,), 0.1, b) + 1,
             routed_up=_normal(seed, 12, (h, lat), 0.02, b),
             residual_norm=_normal(seed, 13, (h,), 0.1, b) + 1,
             residual_proj=_normal(seed, 14, (h,), 0.05, b),
             post_norm=_normal(seed, 15, (h,), 0.1, b) + 1)
    w["router"], w["correction"] = _router(seed, c, b)
    w["shared"] = _shared(seed, c, h)
    return w


def _latent_weights(seed, c):
    h, lat, s = c["hidden"], c["latent"], c["shared_inter"]
    return dict(routed_down=_normal(seed, 10, (lat, h), 0.02),
                routed_norm=_normal(seed, 11, (lat,), 0.1) + 1,
                routed_up=_normal(seed, 12, (h, lat), 0.02),
                shared_gate=_normal(seed, 3, (s, h), 0.02), shared_up=_normal(seed, 4, (s, h), 0.02),
                shared_down=_normal(seed, 5, (h, s), 0.02))


def _routes(seed, c):
    """Routes from the host: distinct experts per token and positive weights that sum to one."""
    r = np.random.RandomState(int(seed) % (1 << 31))
    ids = np.stack([r.permutation(c["experts"])[:c["top_k"]] for _ in range(c["tokens"])])
    w = r.uniform(0.2, 1.0, ids.shape)
    w = (w / w.sum(1, keepdims=True)).astype(np.float32)
    return ids.astype(np.uint32), w


# ---- the calls --------------------------------------------------------------------------------

def _crc32c(k3x_amd, ctx, extent):
    st, v = ctx.crc32c(extent)
    k3x_amd.check(st, "crc32c")
    return v


def _fill_bank(k3x_amd, ctx, seed, c, hidden, shared_inter=0):
    bank = k3x_amd.Bank(ctx, k3x_amd.LayerShape(hidden, c["inter"], c["experts"], shared_inter))
    for e in range(c["experts"]):
        ex = _extents(*_expert(seed, e, hidden, c["inter"]))
        k3x_amd.check(bank.upload_expert_device(e, ex, (3 * e + 1, 3 * e + 2, 3 * e + 3)),
                      "upload expert")
    return bank


def prepare(case, seed):
    import k3x_amd
    c = case
    T, H = c["tokens"], c["hidden"]
    ctx = k3x_amd.Context(0)
    s = dict(k=k3x_amd, kind=c["kind"], ctx=ctx)
    if c["kind"] == "layer":
        bank = _fill_bank(k3x_amd, ctx, seed, c, H, c["shared_inter"])
        w, bias = _router(seed, c)
        gamma = _normal(seed, 6, (H,), 0.1) + 1
        k3x_amd.check(bank.set_router_device(w, bias, gamma), "router")
        if c["shared_inter"]:
            k3x_amd.check(bank.upload_shared(*[_host_bits(m) for m in _shared(seed, c, H)]),
                          "shared expert")
        glu = k3x_amd.GLU_SWIGLU if c["glu"] == "swiglu" else k3x_amd.GLU_SITU
        renorm = k3x_amd.RENORM_FLOAT if c["renorm"] == "float" else k3x_amd.RENORM_DOUBLE
        s.update(bank=bank, x=_normal(seed, 7, (T, H), 1.0, torch.bfloat16),
                 out=torch.empty((T, H), dtype=torch.bfloat16, device=DEV),
                 params=k3x_amd.make_params(T, c["top_k"], c["routed_scale"], EPS, glu, BETA,
                                            LINEAR if c["glu"] == "situ" else None, renorm))
    elif c["kind"] == "official":
        bank = _fill_bank(k3x_amd, ctx, seed, c, c["latent"])
        off = k3x_amd.Official(ctx, bank, H, c["shared_inter"])
        w = _official_weights(seed, c)
        k3x_amd.check(off.upload_ffn(*[_host_bits(w[n]) for n in
                                       ("routed_down", "routed_norm", "routed_up")],
                                     *[_host_bits(m) for m in w["shared"]]), "upload ffn")
        k3x_amd.check(off.upload_route(*[_host_bits(w[n]) for n in
                                         ("residual_norm", "residual_proj", "post_norm",
                                          "router")], w["correction"].cpu().numpy()),
                      "upload route")
        s.update(bank=bank, off=off, tokens=T, prefix=_normal(seed, 7, (T, H), 1.0),
                 residual=_normal(seed, 8, (T, H), 1.0),
                 hidden=torch.empty((T, H), dtype=torch.bfloat16, device=DEV),
                 out=torch.empty((T, H), dtype=torch.bfloat16, device=DEV),
                 params=k3x_amd.make_params(T, c["top_k"], 1.0, OFFICIAL_EPS, k3x_amd.GLU_SITU,
                                            BETA, LINEAR, k3x_amd.RENORM_DOUBLE))
    elif c["kind"] == "latent":
        bank = _fill_bank(k3x_amd, ctx, seed, c, c["latent"])
        ids, contributions = _routes(seed, c)
        s.update(bank=bank, w=_latent_weights(seed, c), x=_normal(seed, 7, (T, H), 1.0),
                 out=torch.empty((T, H), dtype=torch.float32, device=DEV),
                 host_ids=ids, host_contributions=contributions,
                 ids=torch.from_numpy(ids.view(np.int32)).to(DEV),
                 contributions=torch.from_numpy(contributions).to(DEV),
                 params=k3x_amd.make_params(T, c["top_k"], 1.0, EPS, k3x_amd.GLU_SITU, BETA,
                                            LINEAR))
    else:
        bank = k3x_amd.Bank(ctx, k3x_amd.LayerShape(H, c["inter"], c["experts"], 0))
        ids, contributions = _routes(seed, c)
        records = []
        for e in ids[0].tolist():
            ex = _extents(*_expert(seed, e, H, c["inter"]))
            records.append((e, ex, [_crc32c(k3x_amd, ctx, t) for t in ex]))
        s.update(bank=bank, records=records, x=_normal(seed, 7, (T, H), 1.0, torch.bfloat16),
                 out=torch.empty((T, H), dtype=torch.bfloat16, device=DEV),
                 host_ids=ids, host_contributions=contributions,
                 ids=torch.from_numpy(ids.view(np.int32)).to(DEV),
                 contributions=torch.from_numpy(contributions).to(DEV),
                 params=k3x_amd.make_params(T, c["top_k"], 1.0, EPS, k3x_amd.GLU_SWIGLU))
    return s


def run(state):
    s = state
    k, ctx = s["k"], s["ctx"]
    if s["kind"] == "layer":
        k.check(k.moe_forward(ctx, s["bank"], s["params"], s["x"], s["out"]), "moe_forward")
        return s["out"]
    if s["kind"] == "official":
        off = s["off"]
        k.check(off.prepare(s["tokens"], OFFICIAL_EPS, s["prefix"], s["residual"], s["hidden"]),
                "official prepare")
        k.check(off.ffn(s["params"], s["hidden"], s["prefix"], s["out"]), "official ffn")
        return {"hidden": s["hidden"], "out": s["out"]}
    if s["kind"] == "latent":
        k.check(k.resident_moe_layer(ctx, s["bank"], s["w"], s["params"], s["x"], s["ids"],
                                     s["contributions"], s["out"], host_ids=s["host_ids"],
                                     host_contributions=s["host_contributions"]),
                "resident_moe_layer")
        return s["out"]
    for e, ex, crcs in s["records"]:
        k.check(s["bank"].upload_expert_device(e, ex, (3 * e + 1, 3 * e + 2, 3 * e + 3), crcs),
                "upload expert")
    k.check(k.moe_forward_routed(ctx, s["bank"], s["params"], s["x"], s["ids"],
                                 s["contributions"], s["out"], s["host_ids"],
                                 s["host_contributions"]), "moe_forward_routed")
    return s["out"]


# ---- what a call cannot do without ------------------------------------------------------------

def _experts_touched(c):
    """Distinct experts of the case's routes, from a simulation of its router's scores."""
    T, E, K = c["tokens"], c["experts"], c["top_k"]
    r = np.random.RandomState(1)
    if c.get("zipf"):
        bias = 0.45 * np.arange(1, E + 1) ** -1.1
    else:
        bias = 0.1 * r.standard_normal(E)
    logits = r.standard_normal((T, E)) * 0.02 * c["hidden"] ** 0.5
    scores = 1 / (1 + np.exp(-logits)) + bias
    return len(np.unique(np.argpartition(-scores, K - 1, axis=1)[:, :K]))


def work(case):
    c = case
    T, H, I, K, E = c["tokens"], c["hidden"], c["inter"], c["top_k"], c["experts"]
    width = c.get("latent", H)
    expert = 3 * (width * I // 2 + width * I // 32)
    flops = T * K * 6 * width * I
    if c["kind"] == "layer":
        S = c["shared_inter"]
        return {"bytes": _experts_touched(c) * expert + 3 * S * H * 2 + E * H * 4 + 4 * T * H,
                "flops": flops + T * (6 * S * H + 2 * E * H)}
    if c["kind"] == "official":
        S = c["shared_inter"]
        return {"bytes": _experts_touched(c) * expert + (2 * width * H + 3 * S * H) * 2 +
                E * H * 2 + 12 * T * H,
                "flops": flops + T * (4 * width * H + 6 * S * H + 2 * E * H)}
    if c["kind"] == "latent":
        S = c["shared_inter"]
        used = E * (1 - (1 - K / E) ** T)
        return {"bytes": used * expert + (2 * width * H + 3 * S * H) * 4 + 8 * T * H,
                "flops": flops + T * (4 * width * H + 6 * S * H)}
    # Admission: each record read once for its checksum, written once to its slot; then read.
    return {"bytes": 3 * K * expert + 4 * T * H, "flops": flops}


def tolerance(case):
    # About four times what a plain 64-bit computation with the same rounding points differs by
    # (largest of the listed cases and drawn ones).
    if case["kind"] == "latent":
        # fp32 results, experts on bf16 hi + lo halves with fp32 sums: 2.1e-6, max 7.7e-6.
        return {"rel": 8e-6, "max": 3.2e-5}
    if case["kind"] == "official":
        # Chained bf16 roundings, one ulp apart here and there: 1.13e-3, max 2.1e-2.
        return {"rel": 4.5e-3, "max": 8e-2}
    # bf16 outputs and activations one ulp apart here and there: 2.65e-4, max 7.8e-3 (one ulp).
    return {"rel": 1.1e-3, "max": 3.2e-2}


# ---- the same in 64 bits ----------------------------------------------------------------------

_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _dequant(codes, scales, rows, cols):
    lut = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device=codes.device)
    nib = torch.stack([codes & 15, codes >> 4], dim=-1).reshape(rows, cols // 32, 32)
    sc = torch.exp2(scales.double() - 127).reshape(rows, cols // 32, 1)
    return (lut[nib.long()] * sc).reshape(rows, cols)


def _bf(x):
    return x.to(torch.float32).to(torch.bfloat16).double()


def _same(x):
    return x


def _glu(g, u, kind, linear):
    sig = 1 / (1 + torch.exp(-g))
    if kind == "swiglu":
        return g * sig * u
    return BETA * torch.tanh(g / BETA) * sig * (LINEAR * torch.tanh(u / LINEAR) if linear else u)


def _rmsnorm(x, weight, eps):
    """fp32 rounding where the layer has it: the mean square, the inverse and both products."""
    x32 = x.float()
    ms = x.double().square().mean(1, keepdim=True).float()
    inv = 1.0 / torch.sqrt(ms + eps)
    return ((x32 * inv) * weight.float()).to(torch.bfloat16).double()


def _route(xn, w, bias, K, scale):
    logits = (xn @ w.double().t()).float()
    score = 1.0 / (1.0 + torch.exp(-logits.double()).float())
    ids = torch.sort(score + bias, dim=1, descending=True, stable=True).indices[:, :K]
    picked = torch.gather(score, 1, ids).double()
    return ids, picked / picked.sum(1, keepdim=True) * scale


def _mix_experts(seed, c, x, ids, weights, width, kind, linear, act_round, out_round):
    """Sum over slots of weight * expert(x)."""
    acc = torch.zeros((x.shape[0], width), dtype=torch.float64, device=DEV)
    for e in torch.unique(ids).tolist():
        codes, scales = _expert(seed, e, width, c["inter"])
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        gate, up = (_dequant(codes[i], scales[i], c["inter"], width) for i in (0, 1))
        act = act_round(_glu(x[tok] @ gate.t(), x[tok] @ up.t(), kind, linear))
        y = out_round(act @ _dequant(codes[2], scales[2], width, c["inter"]).t())
        acc.index_add_(0, tok, weights[tok, slot].unsqueeze(1) * y)
    return acc


def exact(case, seed):
    c = case
    T, H = c["tokens"], c["hidden"]
    if c["kind"] == "layer":
        w, bias = _router(seed, c)
        gamma = _normal(seed, 6, (H,), 0.1) + 1
        xn = _rmsnorm(_normal(seed, 7, (T, H), 1.0, torch.bfloat16), gamma, EPS)
        ids, weights = _route(xn, w, bias, c["top_k"], c["routed_scale"])
        linear = c["glu"] == "situ"
        out = _mix_experts(seed, c, xn, ids, weights, H, c["glu"], linear, _bf, _same)
        if c["shared_inter"]:
            g, u, d = (m.double() for m in _shared(seed, c, H))
            out += _bf(_glu(xn @ g.t(), xn @ u.t(), c["glu"], linear)) @ d.t()
        return out
    if c["kind"] == "official":
        w = _official_weights(seed, c)
        prefix = _bf(_normal(seed, 7, (T, H), 1.0))
        src = [_bf(_normal(seed, 8, (T, H), 1.0)).float(), prefix.float()]
        score = []
        for v in src:  # the fp32 inverse and normalised row, as the layer documents them
            inv = 1.0 / torch.sqrt(v.double().square().mean(1, keepdim=True).float() + OFFICIAL_EPS)
            score.append(((v * inv).double() * w["residual_norm"].double() *
                          w["residual_proj"].double()).sum(1).float())
        p = torch.softmax(torch.stack(score, 1).double(), 1).float()
        hidden = _rmsnorm(_bf(p[:, :1] * src[0] + p[:, 1:] * src[1]), w["post_norm"], OFFICIAL_EPS)
        ids, weights = _route(hidden, w["router"], w["correction"], c["top_k"], 1.0)
        lat = _bf(hidden @ w["routed_down"].double().t())
        mixed = _bf(_mix_experts(seed, c, lat, ids, weights, c["latent"], "situ", True, _same, _bf))
        normed = _rmsnorm(mixed, w["routed_norm"], OFFICIAL_EPS)
        routed = _bf(normed @ w["routed_up"].double().t())
        g, u, d = (m.double() for m in w["shared"])
        act = _glu(_bf(hidden @ g.t()), _bf(hidden @ u.t()), "situ", True)
        return {"hidden": hidden, "out": prefix + _bf(routed + _bf(act @ d.t()))}
    ids, weights = _routes(seed, c)
    ids = torch.from_numpy(ids.astype(np.int64)).to(DEV)
    weights = torch.from_numpy(weights).to(DEV).double()
    if c["kind"] == "latent":
        w = {n: t.double() for n, t in _latent_weights(seed, c).items()}
        x = _normal(seed, 7, (T, H), 1.0).double()
        lat = x @ w["routed_down"].t()
        mixed = _mix_experts(seed, c, lat, ids, weights, c["latent"], "situ", True, _same, _same)
        normed = mixed / torch.sqrt(mixed.square().mean(1, keepdim=True) + EPS) * w["routed_norm"]
        act = _glu(x @ w["shared_gate"].t(), x @ w["shared_up"].t(), "situ", True)
        return normed @ w["routed_up"].t() + act @ w["shared_down"].t()
    x = _normal(seed, 7, (T, H), 1.0, torch.bfloat16).double()
    return _mix_experts(seed, c, x, ids, weights, H, "swiglu", False, _bf, _same)
