"""Performance cases: the calls a program makes of this package, from one row answered at once to a fit of 10,000 rows.

The network is the full TabICL v2 architecture with random-init weights (`model.FULL_CLASSIFIER`, `FULL_REGRESSOR`,
seed 2), as in bench.py. Tables, fitted caches and queries are synthetic and made from the seed: table columns are
N(0, 1) with every seventh a small integer code; a cache's keys and values are what a layer norm and a projection leave
(a mean of its own per coordinate, spread 0.55), stored in the bundle's chunk records of f32, i16 or i8.

Kinds of case (`op`):

* `predict`: test rows through all three stages against a fitted member, inputs and outputs in host arrays
  (`Gpu.predict`) or, with `dev`, resident on the card (`Gpu.predict_dev`);
* `attend`: one layer's in-context attention of scaled queries over a member's cache (`Gpu.attend_resident_dev`);
* `classes`: a member of more classes than the network's ten: `Gpu.embed` and `Gpu.represent`, then `Gpu.in_context` of
  every problem of the class tree (the host's walk down the tree is not part of the case);
* `fit`: `fit.fit_raw`, a table to its fitted member. f32 and i8 caches: an i16 code is 2^-15 of its chunk's range, so
  that the rounding of any f32 sum before it moves whole codes;
* `quantiles`: a regression member's predicted quantiles read as distributions (`Gpu.quantile_stats_dev`).
"""
import functools
import importlib
import math

import numpy as np
import torch

abi = importlib.import_module("tabicl-anywhere_amd.abi")
fitmod = importlib.import_module("tabicl-anywhere_amd.fit")
hip = importlib.import_module("tabicl-anywhere_amd.hip")
modelmod = importlib.import_module("tabicl-anywhere_amd.model")
planmod = importlib.import_module("tabicl-anywhere_amd.plan")

FORMATS = {"f32": abi.KV_F32, "i16": abi.KV_I16, "i8": abi.KV_I8}
LEVELS = (0.5, 0.025, 0.975, 0.1, 0.9, 0.25, 0.75, 0.01, 0.99, 0.0005, 0.9995)


def listed():
    return [
        # a request answered at once against a resident member: latency
        {"name": "predict_1_f32", "op": "predict", "model": "clf", "n": 1, "rows": 10000, "features": 100, "kv": "f32",
         "chunk": 256, "dev": False},
        # a handful of rows against a small member, odd sizes everywhere
        {"name": "predict_7_i16", "op": "predict", "model": "clf", "n": 7, "rows": 1333, "features": 23, "kv": "i16",
         "chunk": 256, "dev": False},
        # a small batch of a serving loop, the smallest cache format
        {"name": "predict_64_i8", "op": "predict", "model": "clf", "n": 64, "rows": 10000, "features": 100, "kv": "i8",
         "chunk": 256, "dev": True},
        # an ordinary table scored in one call, sizes that divide nothing
        {"name": "predict_777_i16", "op": "predict", "model": "clf", "n": 777, "rows": 3001, "features": 37, "kv": "i16",
         "chunk": 256, "dev": True},
        # the headline batch
        {"name": "predict_2048_f32", "op": "predict", "model": "clf", "n": 2048, "rows": 10000, "features": 100,
         "kv": "f32", "chunk": 256, "dev": True},
        # a wide regression table (200 features, 999 quantiles a row)
        {"name": "predict_500_wide", "op": "predict", "model": "reg", "n": 500, "rows": 5000, "features": 200,
         "kv": "f32", "chunk": 256, "dev": True},
        # the attention hook alone over a long quantised cache
        {"name": "attend_2048_i16", "op": "attend", "model": "clf", "n": 2048, "rows": 20000, "kv": "i16", "chunk": 256},
        # forty classes on a ten-class network: two label digits, a class tree of several problems
        {"name": "classes_40", "op": "classes", "model": "clf", "n": 256, "rows": 2000, "features": 30, "classes": 40,
         "kv": "f32", "chunk": 256},
        # the smallest fits: a few hundred rows
        {"name": "fit_400_i8", "op": "fit", "model": "clf", "rows": 400, "features": 12, "kv": "i8", "chunk": 256},
        # a wide regression fit
        {"name": "fit_1500_wide", "op": "fit", "model": "reg", "rows": 1500, "features": 200, "kv": "f32", "chunk": 256},
        # the headline fit
        {"name": "fit_10000_f32", "op": "fit", "model": "clf", "rows": 10000, "features": 100, "kv": "f32", "chunk": 256},
        # eight members' outputs for 2,048 rows read as distributions
        {"name": "quantiles_16384", "op": "quantiles", "rows": 16384, "quantiles": 999, "levels": 6},
    ]


def draw(rng):
    def between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["predict", "predict", "predict", "attend", "classes", "fit", "fit", "quantiles"])
    kv, model, chunk = rng.choice(["f32", "i16", "i8"]), rng.choice(["clf", "clf", "reg"]), rng.choice([256, 256, 256, 100])
    if op == "predict":
        n, features = between(1, 2048), between(5, 200)
        n = min(n, 204800 // features)
        return {"op": op, "model": model, "n": n, "rows": between(300, 10000), "features": features, "kv": kv,
                "chunk": chunk, "dev": rng.random() < 0.5}
    if op == "attend":
        n, rows = between(1, 2048), between(1000, 50000)
        return {"op": op, "model": "clf", "n": min(n, 40960000 // rows), "rows": rows, "kv": kv, "chunk": chunk}
    if op == "classes":
        return {"op": op, "model": "clf", "n": between(10, 300), "rows": between(500, 3000), "features": between(5, 40),
                "classes": rng.randint(11, 60), "kv": kv, "chunk": 256}
    if op == "fit":
        features = between(5, 200)
        return {"op": op, "model": model, "rows": min(between(300, 10000), 600000 // features), "features": features,
                "kv": rng.choice(["f32", "i8"]), "chunk": chunk}
    return {"op": op, "rows": between(200, 16384), "quantiles": rng.choice([99, 500, 999, 999]), "levels": rng.randint(1, 11)}


# ---- what a program has in hand ---------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def network(kind):
    return modelmod.Model.random(modelmod.FULL_CLASSIFIER if kind == "clf" else modelmod.FULL_REGRESSOR, seed=2)


@functools.lru_cache(maxsize=None)
def card():
    return hip.Gpu(0)


@functools.lru_cache(maxsize=None)
def weights(kind):
    return card().weights(network(kind))


def table(rows, features, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, features)).astype(np.float32)
    x[:, ::7] = rng.integers(0, 12, x[:, ::7].shape).astype(np.float32) / 3.5 - 1.5
    return x


def targets(case, seed):
    rng = np.random.default_rng([seed, 1])
    if case["model"] == "reg":
        return rng.standard_normal(case["rows"]).astype(np.float32)
    classes = case.get("classes", 10)
    y = rng.integers(0, classes, case["rows"])
    y[:classes] = np.arange(classes)  # every class occurs
    return y.astype(np.float32)


def generator(*key):
    return torch.Generator(device="cuda").manual_seed(hash(key) & 0x7FFFFFFF)


def layer_values(d, rows, key):
    """A layer's keys and values [rows][2d] as a fit would form them, before they are stored."""
    g = generator(*key)
    mean = torch.randn(2 * d, device="cuda", generator=g) * 0.3
    return torch.randn(rows, 2 * d, device="cuda", generator=g) * 0.55 + mean


def chunk_records(kv, chunk, fmt):
    """The stored records (uint8) of keys and values [rows][2d]: per chunk its scales, then codes by coordinate."""
    parts = []
    full = kv.shape[0] // chunk
    for part in (kv[:full * chunk].view(full, chunk, -1), kv[full * chunk:].unsqueeze(0)):
        if part.numel() == 0:
            continue
        c = part.transpose(1, 2).contiguous()  # [chunks][2d][rows of a chunk]
        if fmt == "f32":
            parts.append(c.view(c.shape[0], -1).view(torch.uint8).reshape(-1))
            continue
        top, kind = (32767.0, torch.int16) if fmt == "i16" else (127.0, torch.int8)
        big = c.abs().amax(2)
        s = torch.where(big > 0, big / top, torch.ones_like(big))
        v = c * (1.0 / s)[..., None]
        codes = torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v)).clamp(-top - 1, top).to(kind)
        codes = codes.view(c.shape[0], -1).view(torch.uint8)
        parts.append(torch.cat([s.view(torch.uint8).view(c.shape[0], -1), codes.view(c.shape[0], -1)], 1).reshape(-1))
    return torch.cat(parts)


def stored_values(rec, rows, chunk, fmt, d):
    """Records back to keys and values [rows][2d] in 64 bits: what a prediction reads."""
    out, at = [], 0
    for rc in [chunk] * (rows // chunk) + ([rows % chunk] if rows % chunk else []):
        size = abi.kv_record(FORMATS[fmt], d, rc)
        c, at = rec[at:at + size].clone(), at + size
        if fmt == "f32":
            out.append(c.view(torch.float32).double().view(2 * d, rc).T)
        else:
            s = c[:8 * d].clone().view(torch.float32).double()
            codes = c[8 * d:].clone().view(torch.int16 if fmt == "i16" else torch.int8).double()
            out.append((codes.view(2 * d, rc) * s[:, None]).T)
    return torch.cat(out)


def query_scales(net, rows):
    return np.stack([fitmod.query_scale(b, rows) for b in net.icl]).astype(np.float32)


def column_cache(net, features, digits, seed):
    g = generator(seed, 77)
    shape = (features, digits, len(net.col_a2), 2, net.e, net.inds)
    mean = torch.randn(shape[:-1] + (1,), device="cuda", generator=g) * 0.3
    return torch.randn(shape, device="cuda", generator=g) * 0.55 + mean


def member(case, rows, seed, node=0):
    """A member's in-context problem on the card, loaded from its stored records."""
    net, fmt = network(case["model"]), case["kv"]
    layers = [chunk_records(layer_values(net.d, rows, (seed, node, l)), case["chunk"], fmt).cpu().numpy()
              for l in range(net.icl_layers)]
    return card().load(weights(case["model"]), FORMATS[fmt], rows, case["chunk"], layers, query_scales(net, rows))


def plan_of(case, seed):
    net = network(case["model"])
    return planmod.Plan.new(net.max_classes, targets(case, seed), case.get("classes", 10))


def queries(case, seed):
    return torch.randn(case["n"], network(case["model"]).d, device="cuda", generator=generator(seed, 5)) * 0.2


def outputs_of(case):
    return network(case["model"]).outputs


def quantile_rows(case, seed):
    g = generator(seed, 9)
    q = torch.randn(case["rows"], case["quantiles"], device="cuda", generator=g)
    spread = torch.rand(case["rows"], 1, device="cuda", generator=g) * 3.0 + 0.2
    # a network's quantiles come nearly in order
    ramp = torch.linspace(-2.0, 2.0, case["quantiles"], device="cuda")
    return ((q * 0.1 + ramp) * spread + 1.0).contiguous()


def prepare(case, seed):
    op = case["op"]
    s = {"case": case, "gpu": card()}
    if op == "quantiles":
        s["q"] = quantile_rows(case, seed)
        s["levels"] = np.array(LEVELS[:case["levels"]], np.float32)
        s["out"] = torch.empty(case["rows"], 3 + case["levels"], device="cuda")
        torch.cuda.synchronize()
        return s
    net = network(case["model"])
    s["weights"] = weights(case["model"])
    if op == "fit":
        s["x"], s["y"] = table(case["rows"], case["features"], seed), targets(case, seed)
        s["classes"] = 10 if case["model"] == "clf" else net.outputs
        return s
    if op == "attend":
        s["member"] = member(case, case["rows"], seed)
        s["q"] = queries(case, seed)
        s["out"] = torch.empty_like(s["q"])
        torch.cuda.synchronize()
        return s
    x = table(case["n"], case["features"], seed + 1000003)
    if op == "classes":
        plan = plan_of(case, seed)
        s["members"] = [member(case, len(node.y), seed, i) for i, node in enumerate(plan.nodes)]
        s["outs"] = [node.k for node in plan.nodes]
        digits = len(plan.bases)
        s["members"][0].set_columns(column_cache(net, case["features"], digits, seed).cpu().numpy(), case["features"], digits)
        s["x"] = x
        return s
    s["member"] = member(case, case["rows"], seed)
    s["member"].set_columns(column_cache(net, case["features"], 1, seed).cpu().numpy(), case["features"], 1)
    if case["dev"]:
        s["x"] = torch.from_numpy(x).cuda()
        s["out"] = torch.empty(case["n"], net.outputs, device="cuda")
        torch.cuda.synchronize()
    else:
        s["x"] = x
    return s


def record_arrays(records, rows, chunk, fmt, d):
    """A layer's records as arrays of what they hold (views): f32 values, or per chunk its scales and its codes."""
    if fmt == "f32":
        return [records.view(np.float32)]
    full, size = rows // chunk, abi.kv_record(FORMATS[fmt], d, chunk)
    parts = [records[:full * size].reshape(full, size)] if full else []
    if rows % chunk:
        parts.append(records[full * size:].reshape(1, -1))
    return [a for p in parts for a in (p[:, :8 * d].view(np.float32), p[:, 8 * d:].view(np.int8))]


def run(state):
    case, gpu = state["case"], state["gpu"]
    op = case["op"]
    if op == "predict":
        if not case["dev"]:
            return gpu.predict(state["weights"], state["member"], state["x"], outputs_of(case))
        gpu.predict_dev(state["weights"], state["member"], state["x"].data_ptr(), case["n"], outputs_of(case),
                        state["out"].data_ptr())
        return state["out"]
    if op == "attend":
        gpu.attend_resident_dev(state["member"], 0, state["q"].data_ptr(), case["n"], state["out"].data_ptr())
        return state["out"]
    if op == "quantiles":
        gpu.quantile_stats_dev(state["q"].data_ptr(), case["rows"], case["quantiles"], state["levels"],
                               state["out"].data_ptr())
        return state["out"]
    if op == "classes":
        w = state["weights"]
        rep = gpu.represent(w, gpu.embed(w, state["members"][0], state["x"]))
        return [gpu.in_context(w, vm, rep, k) for vm, k in zip(state["members"], state["outs"])]
    fitted = fitmod.fit_raw(gpu, state["weights"], state["x"], state["y"], state["classes"], case["chunk"],
                            FORMATS[case["kv"]])
    d = network(case["model"]).d
    return {"columns": fitted.col_kv, "scales": fitted.scales[0],
            "layers": [record_arrays(r, case["rows"], case["chunk"], case["kv"], d) for r in fitted.layers[0]]}


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def cache_bytes(net, rows, kv, chunk):
    size = {"f32": 4, "i16": 2, "i8": 1}[kv]
    return 2 * rows * net.d * size + (-(-rows // chunk) * 8 * net.d if size < 4 else 0)


def floats_of(blocks, query_only=False):
    return sum(a.size // 3 if query_only and k in ("in_w", "in_b") else a.size for b in blocks for k, a in b.t.items())


def row_flops(net, T):
    e, full = net.e, len(net.row) - 1
    return 2 * (full * T * (8 * e * e + 2 * T * e) + 2 * e * e * T + net.cls * (6 * e * e + 2 * T * e))


def stage_flops(net, rows, outputs):
    d, ff = net.d, net.icl[0].ff
    layer = 4 * rows * d + 2 * (2 * d * d + 2 * d * ff + 2 * d * 64)
    return net.icl_layers * layer + 2 * (net.dec_hidden * d + outputs * net.dec_hidden)


def work(case):
    op = case["op"]
    if op == "quantiles":
        # a comparison sort's n log2 n, and the sums
        n = case["quantiles"]
        return {"bytes": 4.0 * case["rows"] * (n + 3 + case["levels"]), "flops": case["rows"] * n * (math.log2(n) + 4.0)}
    net, rows = network(case["model"]), case["rows"]
    d, e, inds = net.d, net.e, net.inds
    if op == "attend":
        return {"bytes": cache_bytes(net, rows, case["kv"], case["chunk"]) + 8.0 * case["n"] * d,
                "flops": 4.0 * case["n"] * rows * d}
    features, T = case["features"], net.cls + case["features"]
    if op == "fit":
        L, ff = net.icl_layers, net.icl[0].ff
        nbytes = (4.0 * (floats_of(net.col_a1 + net.col_a2 + net.row + net.icl) + rows * features)
                  + L * cache_bytes(net, rows, case["kv"], case["chunk"]) + 4.0 * features * 3 * 2 * e * inds)
        cells = rows * features * 3.0 * (16 * e * e + 8 * inds * e)
        layers = rows * (L * 4.0 * d * d + (L - 1) * (4.0 * rows * d + 2 * (2 * d * d + 2 * d * ff + 2 * d * 64)))
        return {"bytes": nbytes, "flops": cells + rows * float(row_flops(net, T)) + layers}
    w = 4.0 * (floats_of(net.col_a2 + net.icl, True) + floats_of(net.row) + net.dec_hidden * (d + outputs_of(case)))
    cell = 3.0 * (12 * e * e + 4 * inds * e)
    if op == "classes":
        plan = plan_of(case, 1)
        digits = len(plan.bases)
        nodes = [(len(node.y), node.k) for node in plan.nodes]
    else:
        digits, nodes = 1, [(rows, outputs_of(case))]
    nbytes = (w + 4.0 * features * digits * 3 * 2 * e * inds
              + sum(net.icl_layers * cache_bytes(net, r, case["kv"], case["chunk"]) + 4.0 * case["n"] * k for r, k in nodes)
              + 4.0 * case["n"] * features)
    flops = case["n"] * (features * digits * cell + row_flops(net, T) + sum(stage_flops(net, r, k) for r, k in nodes))
    return {"bytes": nbytes, "flops": float(flops)}


def tolerance(case):
    # 32-bit arithmetic throughout: every case measured 1e-7 to 5e-7 from its values in 64 bits, the deepest (twelve
    # layers) the most. An i8 code turns over where its value lies within that of a half: 4e-7 / (1 / 127) of them.
    return {"rel": 2e-6, "differ": 5e-4} if case["op"] == "fit" else {"rel": 2e-6}


# ---- the same in 64 bits, in plain torch ---------------------------------------------------------------------------
def f64(a):
    return torch.as_tensor(a, device="cuda").double()


def norm(x, w, b):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), f64(w), f64(b), 1e-5)


def linear(x, w, b):
    out = b.shape[0]
    return x @ f64(w).view(out, -1).T + f64(b)


def gelu(x):
    return torch.nn.functional.gelu(x)


def feed_forward(b, x):
    t = b.t
    return x + linear(gelu(linear(norm(x, t["n2w"], t["n2b"]), t["l1w"], t["l1b"])), t["l2w"], t["l2b"])


def split_heads(x, heads):
    return x.unflatten(-1, (heads, x.shape[-1] // heads)).transpose(-2, -3)


def softmax_average(q, k, v):
    """q [..][nq][hd], k and v [..][n][hd], queries already scaled; over a bounded number of queries at a time."""
    step = max(1, int(2.5e8 // max(1, k.shape[-2] * math.prod(k.shape[:-2]))))
    return torch.cat([torch.softmax(q[..., i:i + step, :] @ k.transpose(-1, -2), -1) @ v
                      for i in range(0, q.shape[-2], step)], -2)


def scaled_query(b, x, scale):
    t, d = b.t, b.d
    q = linear(norm(x, t["n1w"], t["n1b"]), t["in_w"].reshape(3 * d, d)[:d], t["in_b"][:d])
    if not b.ss_hidden:
        return q * scale
    qh = q.unflatten(-1, (b.heads, b.hd))
    m = linear(gelu(linear(qh, t["q0w"], t["q0b"])), t["q2w"], t["q2b"])
    return (qh * (1.0 + torch.tanh(m))).flatten(-2) * scale


def exact_scale(b, n):
    inv = 1.0 / math.sqrt(b.hd)
    if not b.ss_hidden:
        return torch.full((b.d,), inv, device="cuda", dtype=torch.float64)
    t = b.t
    return linear(gelu(f64(t["b0w"]) * math.log(max(n, 1)) + f64(t["b0b"])), t["b2w"], t["b2b"]) * inv


def key_values(b, x):
    t, d = b.t, b.d
    return linear(norm(x, t["n1w"], t["n1b"]), t["in_w"].reshape(3 * d, d)[d:], t["in_b"][d:])


def block_over(b, x, scale, kv):
    """x [..][n][d] through block b over keys and values kv [..][keys][2d]."""
    k, v = kv[..., :b.d], kv[..., b.d:]
    a = softmax_average(split_heads(scaled_query(b, x, scale), b.heads), split_heads(k, b.heads), split_heads(v, b.heads))
    return feed_forward(b, x + linear(a.transpose(-2, -3).flatten(-2), b.t["out_w"], b.t["out_b"]))


def input_cells(net, x):
    """[features][rows][e]"""
    x = f64(x)
    F = x.shape[1]
    vals = torch.stack([x[:, [(g + (1 << k)) % F for g in range(F)]] for k in range(net.group)], -1)
    return linear(vals, net.t["in_w"], net.t["in_b"]).transpose(0, 1)


def embedding(net, table_, y, width):
    t = f64(net.t[table_])
    if net.max_classes:
        return t.view(-1, width)[torch.as_tensor(y, device="cuda").long()]
    return t.view(2, width)[0] * f64(y)[:, None] + t.view(2, width)[1]


def exact_rows(net, cells):
    """Representations [rows][d] of cells [features][rows][e]."""
    out = []
    T, hd = net.cls + cells.shape[0], net.e // net.row_heads
    ang = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * f64(net.t["rope_freqs"])[None, :]
    cos, sin = torch.cos(ang), torch.sin(ang)

    def turn(z, n):
        a, b = z[..., :hd // 2], z[..., hd // 2:]
        return torch.cat([a * cos[:n] - b * sin[:n], b * cos[:n] + a * sin[:n]], -1)

    step = max(1, 60000 // T)
    for r0 in range(0, cells.shape[1], step):
        part = cells[:, r0:r0 + step].transpose(0, 1)
        cls = f64(net.t["cls_tokens"]).view(1, net.cls, net.e).expand(part.shape[0], -1, -1)
        x = torch.cat([cls, part], 1)
        for i, b in enumerate(net.row):
            nq = net.cls if i + 1 == len(net.row) else T
            t, e = b.t, net.e
            n1 = norm(x, t["n1w"], t["n1b"])
            w, bias = t["in_w"].reshape(3 * e, e), t["in_b"]
            q, k, v = (split_heads(linear(n1[:, :m], w[j * e:(j + 1) * e], bias[j * e:(j + 1) * e]), b.heads)
                       for j, m in enumerate((nq, T, T)))
            a = softmax_average(turn(q, nq) / math.sqrt(hd), turn(k, T), v)
            x = feed_forward(b, x[:, :nq] + linear(a.transpose(1, 2).flatten(-2), t["out_w"], t["out_b"]))
        out.append(norm(x, net.t["out_lnw"], net.t["out_lnb"]).flatten(-2))
    return torch.cat(out)


def exact_representations(net, case, seed, digits):
    cells = input_cells(net, table(case["n"], case["features"], seed + 1000003))
    col = column_cache(net, case["features"], digits, seed).double()
    total = 0.0
    for dg in range(digits):
        x = cells
        for i, b in enumerate(net.col_a2):
            kv = col[:, dg, i].flatten(1, 2).transpose(1, 2)  # [features][inds][2e]
            x = torch.cat([block_over(b, x[g:g + 10], 1.0 / math.sqrt(b.hd), kv[g:g + 10])
                           for g in range(0, x.shape[0], 10)])
        total = total + x
    return exact_rows(net, total / digits)


def exact_stage(net, case, h, rows, seed, node, outputs):
    scales = f64(query_scales(net, rows))
    for l, b in enumerate(net.icl):
        rec = chunk_records(layer_values(net.d, rows, (seed, node, l)), case["chunk"], case["kv"])
        h = block_over(b, h, scales[l], stored_values(rec, rows, case["chunk"], case["kv"], net.d))
    t = net.t
    hid = gelu(linear(norm(h, t["lnw"], t["lnb"]), t["dec0w"], t["dec0b"]))
    return linear(hid, t["dec2w"], t["dec2b"])[:, :outputs].cpu().numpy()


def exact_fit(case, seed):
    net, rows = network(case["model"]), case["rows"]
    y, e, d = targets(case, seed), net.e, net.d
    cells = input_cells(net, table(rows, case["features"], seed)) + embedding(net, "col_y", y, e)
    col = []
    for g in range(case["features"]):
        x, blocks = cells[g], []
        for i, (a1, a2) in enumerate(zip(net.col_a1, net.col_a2)):
            ind = f64(net.t["col_ind"]).view(len(net.col_a1), net.inds, e)[i]
            ind = block_over(a1, ind, exact_scale(a1, rows), key_values(a1, x))
            kv = key_values(a2, ind)
            blocks.append(kv.T.reshape(2, e, net.inds))
            x = block_over(a2, x, 1.0 / math.sqrt(a2.hd), kv)
        col.append(torch.stack(blocks))
        cells[g] = x
    h = exact_rows(net, cells) + embedding(net, "icl_y", y, d)
    layers, scales = [], []
    for l, b in enumerate(net.icl):
        kv, scale = key_values(b, h), exact_scale(b, rows)
        scales.append(scale)
        if case["kv"] == "f32":
            chunks = [kv[i:i + case["chunk"]].T.reshape(-1) for i in range(0, rows, case["chunk"])]
            layers.append([torch.cat(chunks).cpu().numpy()])
        else:
            layers.append([None] * len(record_arrays(np.zeros(abi.layer_bytes(FORMATS[case["kv"]], rows, case["chunk"], d),
                                                              np.uint8), rows, case["chunk"], case["kv"], d)))
        if l + 1 < net.icl_layers:
            h = block_over(b, h, scale, kv)
    return {"columns": torch.stack(col)[:, None].cpu().numpy(), "scales": torch.stack(scales).cpu().numpy(), "layers": layers}


def exact_quantiles(case, seed):
    q = quantile_rows(case, seed).double().sort(1).values
    n = case["quantiles"]
    k = max(min(20, n // 4), 1)
    lv = torch.arange(1, n + 1, device="cuda", dtype=torch.float64) / (n + 1)

    def tail(xs, ys):
        dx = xs - xs.mean()
        return ((dx * (ys - ys.mean(1, keepdim=True))).mean(1) / dx.square().mean().clamp(min=1e-6)).abs().clamp(0.01, 100.0)

    left, right = tail(lv[:k].log(), q[:, :k]), tail((1.0 - lv[-k:]).log(), q[:, -k:])
    out = [q.mean(1), q.var(1)]
    for a in (0.5,) + tuple(float(np.float32(v)) for v in LEVELS[:case["levels"]]):
        if a < lv[0]:
            out.append(q[:, 0] + left * (math.log(a) - lv[0].log()))
        elif a > lv[-1]:
            out.append(q[:, -1] - right * (math.log(1.0 - a) - (1.0 - lv[-1]).log()))
        else:
            i = min(max(int(math.floor(a * (n + 1))) - 1, 0), n - 2)
            out.append(q[:, i] + (a * (n + 1) - 1 - i) * (q[:, i + 1] - q[:, i]))
    return torch.stack(out, 1).cpu().numpy()


def exact(case, seed):
    op = case["op"]
    if op == "quantiles":
        return exact_quantiles(case, seed)
    if op == "fit":
        return exact_fit(case, seed)
    net = network(case["model"])
    if op == "attend":
        rec = chunk_records(layer_values(net.d, case["rows"], (seed, 0, 0)), case["chunk"], case["kv"])
        kv = stored_values(rec, case["rows"], case["chunk"], case["kv"], net.d)
        k, v = split_heads(kv[:, :net.d], net.icl_heads), split_heads(kv[:, net.d:], net.icl_heads)
        q = split_heads(queries(case, seed).double(), net.icl_heads)
        return softmax_average(q, k, v).transpose(0, 1).flatten(-2).cpu().numpy()
    if op == "classes":
        plan = plan_of(case, seed)
        rep = exact_representations(net, case, seed, len(plan.bases))
        return [exact_stage(net, case, rep, len(node.y), seed, i, node.k) for i, node in enumerate(plan.nodes)]
    rep = exact_representations(net, case, seed, 1)
    return exact_stage(net, case, rep, case["rows"], seed, 0, outputs_of(case))
