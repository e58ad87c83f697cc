"""What this framework's users have it do, as cases that can be timed.

Each case is one pass through the public Python entry points on one GPU:
KVCache / PagedKVCache appends, AdaptiveAttention.run and its fused decode
steps, at the head shapes and sizes of this repository's own configurations,
tests and benchmark. Four kinds:

  decode   one new token of one layer through the fused append + decode step
           (optionally with RoPE, or with the Qwen3 q/k RMSNorm and RoPE; on a
           contiguous or a paged cache), called eagerly
  step     the decode step of a whole model (all layers), captured once in a
           HIP graph as an engine does, replayed
  attend   n_new tokens of one layer: KVCache.append, then
           AdaptiveAttention.run (prefill, chunked prefill, verification of
           speculated tokens)
  ingest   the RoPE (and q/k-norm) + FP8 append of a prefill chunk, without
           the attention
"""
import math

import torch

import runtherder_amd as R

DEV = "cuda:0"
EPS = 1e-6
THETA = 500000.0

# (q heads, kv heads, head_dim): the head shapes of the repository's
# configurations and tests.
H24, H32, H64, MHA, G7, D64, D256 = ((24, 8, 128), (32, 8, 128), (64, 8, 128), (16, 16, 128),
                                     (28, 4, 128), (32, 8, 64), (16, 4, 256))
MOST_FLOPS = 8.7e12   # of a drawn case: that of the largest listed one
BLOCK = 64            # positions per block of a paged cache


def _case(name, kind, heads, clen, n=1, extra="", paged=False, layers=1):
    c = {"kind": kind, "hq": heads[0], "hkv": heads[1], "d": heads[2], "clen": clen, "n": n,
         "extra": extra, "paged": paged, "layers": layers}
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # A chat's decode early on: the smallest call, all launch and latency.
        _case("decode_511", "decode", H24, 510),
        # The benchmark's headline: a 28-layer model's decode step at 8K,
        # replayed as the engine's HIP graph.
        _case("step28_8196", "step", H24, 8195, layers=28),
        # Decode at a long context with the Qwen3 order and a paged cache, as
        # a server holds it.
        _case("decode_qknorm_paged_32k", "decode", H32, 32767, extra="qk_norm", paged=True),
        # The largest decode of the configurations: 128K of context.
        _case("decode_128k", "decode", H32, 131071),
        # Verification of 8 speculated tokens after 8K of context.
        _case("verify8_8k", "attend", H24, 8192, n=8),
        # A short user turn after a long conversation.
        _case("chunk64_32k", "attend", H32, 32768, n=64),
        # A longer, ragged turn after a long conversation.
        _case("chunk250_32k", "attend", H32, 32768, n=250),
        # An ordinary prompt (the repository's 1021-token configuration).
        _case("prefill_1021", "attend", H24, 0, n=1021),
        # Long prompts.
        _case("prefill_4096", "attend", H32, 0, n=4096),
        _case("prefill_16384", "attend", H32, 0, n=16384),
        # A chunk of a 128K prompt's chunked prefill, the last one.
        _case("chunk4096_128k", "attend", H32, 126976, n=4096),
        # What precedes a 4K prefill's attention in the Qwen3 order: q/k norm,
        # RoPE and the append of K and V.
        _case("ingest_qknorm_4096", "ingest", H32, 0, n=4096, extra="qk_norm"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["decode", "decode", "few", "chunk", "chunk", "prefill", "prefill", "ingest"])
    if what == "decode":
        heads = rng.choice([H24, H32, H32, H64, MHA, G7, D64, D256])
        return _case(None, "decode", heads, _log_int(rng, 30, 131071),
                     extra=rng.choice(["", "rope", "qk_norm"]), paged=rng.random() < 0.4)
    if what == "few":
        heads = rng.choice([H24, H32, H64, G7, D64, D256])
        return _case(None, "attend", heads, _log_int(rng, 100, 65536), n=rng.randint(2, 80),
                     paged=rng.random() < 0.3)
    heads = rng.choice([H24, H32, H32, H64, MHA, G7])
    if what == "chunk":
        n, clen = _log_int(rng, 81, 4096), _log_int(rng, 500, 126976)
    elif what == "prefill":
        n, clen = _log_int(rng, 17, 16384), 0
    else:
        return _case(None, "ingest", heads, rng.choice([0, 1000]), n=_log_int(rng, 1, 8192),
                     extra=rng.choice(["rope", "qk_norm"]))
    while 4.0 * heads[0] * heads[2] * n * (clen + (n + 1) / 2) > MOST_FLOPS:
        n = n * 3 // 4
    return _case(None, "attend", heads, clen, n=n, paged=rng.random() < 0.3)


# ---- inputs ------------------------------------------------------------------

def _tokens(case, seed, layer, what):
    """(q, k, v) bf16 of the new tokens (what "new") or (k, v) of the cached
    ones ("old"). Queries and values are unit normals; key channels differ in
    size, as a trained model's do, so that the attention is neither uniform
    nor a single key."""
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1000003 * seed + 1009 * layer + (1 if what == "new" else 2))
    gain = torch.exp(0.5 * torch.randn((hkv, d), generator=gen, device=DEV))

    def normal(n, h):
        return torch.randn((n, h, d), generator=gen, device=DEV)

    n = case["n"] if what == "new" else case["clen"]
    k = (normal(n, hkv) * gain).to(torch.bfloat16)
    v = normal(n, hkv).to(torch.bfloat16)
    return (normal(n, hq).to(torch.bfloat16), k, v) if what == "new" else (k, v)


def _gains(case, seed):
    """q_norm and k_norm weights [head_dim]."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(77 + seed)
    return [(1.0 + 0.2 * torch.randn(case["d"], generator=gen, device=DEV)).to(torch.bfloat16)
            for _ in range(2)]


def _inv_freq(case):
    i = torch.arange(case["d"] // 2, device=DEV, dtype=torch.float64)
    return (THETA ** (-2.0 * i / case["d"])).to(torch.float32)


def _block_table(case, seed):
    blocks = (case["clen"] + case["n"] + BLOCK - 1) // BLOCK
    gen = torch.Generator(device=DEV)
    gen.manual_seed(13 + seed)
    return torch.randperm(blocks, generator=gen, device=DEV).to(torch.int32)


def _int(v):
    return torch.tensor([v], dtype=torch.int32, device=DEV)


def prepare(case, seed):
    hq, hkv, d, n, clen = (case[x] for x in ("hq", "hkv", "d", "n", "clen"))
    layers = case["layers"]
    s = {"case": case, "pos": _int(clen), "n": n, "backend": R.make_attention_backend(
        R.BackendKind.Adaptive, R.AttnConfig.for_heads(hq, hkv, d))}
    table = _block_table(case, seed) if case["paged"] else None
    if table is not None:
        cache = R.PagedKVCache(layers, len(table), BLOCK, hkv, d, device=DEV)
    else:
        cache = R.KVCache(layers, clen + n, hkv, d, device=DEV)
    # Rows that nobody writes (a paged cache's last block) hold zeros, so that
    # whole slabs compare.
    for t in (cache.k, cache.v, cache.k_scale, cache.v_scale):
        t.zero_()
    zero = _int(0)
    s.update(cache=cache, table=table, q=[], k=[], v=[],
             out=torch.empty((layers, n, hq, d), dtype=torch.bfloat16, device=DEV))
    for layer in range(layers):
        if clen:
            k, v = _tokens(case, seed, layer, "old")
            if table is not None:
                cache.append(layer, k, v, clen, zero, table)
            else:
                cache.append(layer, k, v, clen, zero)
        q, k, v = _tokens(case, seed, layer, "new")
        s["q"].append(q)
        s["k"].append(k)
        s["v"].append(v)
    if case["kind"] in ("decode", "step"):
        s["slabs"] = [cache.slabs(i, table) if table is not None else cache.slabs(i)
                      for i in range(layers)]
    elif case["kind"] == "attend":
        s["view"] = cache.view(0, table) if table is not None else cache.view(0)
    if case["extra"]:
        s["positions"] = torch.arange(clen, clen + n, dtype=torch.int32, device=DEV)
        s["inv_freq"] = _inv_freq(case)
    if case["extra"] == "qk_norm":
        s["q_norm"], s["k_norm"] = _gains(case, seed)
    # What a pass writes: the new tokens' cache rows (a paged cache: the slabs).
    first = 0 if table is not None else clen
    s["new"] = [t[:, first:] for t in (cache.k, cache.v, cache.k_scale, cache.v_scale)]
    if case["kind"] == "step":
        def one_step():
            for i in range(layers):
                s["backend"].run_decode_append(s["out"][i, 0], s["q"][i][0], s["slabs"][i],
                                               s["k"][i], s["v"][i], s["pos"])

        one_step()
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            one_step()
        s["out"].zero_()
    return s


# ---- one pass ----------------------------------------------------------------

def run(s):
    case = s["case"]
    kind, extra = case["kind"], case["extra"]
    if kind == "step":
        s["graph"].replay()
    elif kind == "decode":
        args = (s["out"], s["q"][0], s["slabs"][0], s["k"][0], s["v"][0])
        if extra == "rope":
            s["backend"].run_decode_rope_append(*args, s["positions"], s["inv_freq"], s["pos"])
        elif extra == "qk_norm":
            s["backend"].run_decode_qk_norm_rope_append(*args, s["q_norm"], s["k_norm"], EPS,
                                                        s["positions"], s["inv_freq"], s["pos"])
        else:
            s["backend"].run_decode_append(*args, s["pos"])
    elif kind == "attend":
        if s["table"] is not None:
            s["cache"].append(0, s["k"][0], s["v"][0], s["n"], s["pos"], s["table"])
        else:
            s["cache"].append(0, s["k"][0], s["v"][0], s["n"], s["pos"])
        s["backend"].run(s["out"], s["q"][0], s["view"], s["n"], s["pos"])
    elif extra == "rope":
        s["cache"].append_rope(0, s["q"][0], s["k"][0], s["v"][0], s["n"], s["positions"],
                               s["inv_freq"], s["pos"], case["hq"])
    else:
        s["cache"].append_qk_norm_rope(0, s["q"][0], s["k"][0], s["v"][0], s["n"], s["q_norm"],
                                       s["k_norm"], EPS, s["positions"], s["inv_freq"], s["pos"],
                                       case["hq"])
    # The ingest rotates q in place: it is an output there.
    return {"out": s["q"][0] if kind == "ingest" else s["out"], "k": s["new"][0],
            "v": s["new"][1], "k_scale": s["new"][2], "v_scale": s["new"][3]}


def work(case):
    hq, hkv, d, n, clen = (case[x] for x in ("hq", "hkv", "d", "n", "clen"))
    new = n * hkv * (d * 4 + d * 2 + 8)          # k, v in (bf16), codes and scales out
    q_out = n * hq * d * 4                       # q in, out (or the rotated q) out
    if case["kind"] == "ingest":
        return {"bytes": new + q_out, "flops": 0}
    cached = clen * hkv * (2 * d + 8)
    pairs = n * clen + n * (n + 1) // 2
    return {"bytes": case["layers"] * (cached + new + q_out),
            "flops": case["layers"] * 4 * hq * d * pairs}


def tolerance(case):
    if case["kind"] == "ingest":
        # q to bf16 of an exactly rounded rotation; codes and scales alike.
        return {"rel": 1e-4, "max": 0.02}
    return {"rel": 1e-2, "max": 0.1}


# ---- the same in 64 bits -------------------------------------------------------

def _rms(x, g):
    x = x.double()
    return (x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)) * g.double()


def _rope(x, case, first):
    """Rotate-half RoPE; the angle is the fp32 product the engine takes."""
    d = case["d"]
    pos = torch.arange(first, first + x.shape[0], device=DEV).to(torch.float32)
    a = (pos[:, None] * _inv_freq(case)[None]).double()[:, None]
    x = x.double()
    lo, hi = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([lo * torch.cos(a) - hi * torch.sin(a),
                      hi * torch.cos(a) + lo * torch.sin(a)], -1)


def _quantize(x):
    """(codes as float64, scale fp32) of the FP8 cache format: scale = amax /
    448 per row, codes = E4M3(x * (448 / amax))."""
    x = x.float()
    amax = x.abs().amax(-1)
    inv = torch.where(amax > 0, 448.0 / amax, torch.zeros_like(amax))
    codes = (x * inv[..., None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return codes.double(), amax / 448.0


def _attend(q, k, v, case):
    """q [n, hq, d], k and v [total, hkv, d], all float64."""
    n, hq, d = q.shape
    total, hkv = k.shape[:2]
    group, clen = hq // hkv, case["clen"]
    out = torch.empty_like(q)
    step = max(1, int(6e8) // (total * group))   # rows at once: about 5 GB
    for h in range(hkv):
        kt, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for a in range(0, n, step):
            b = min(n, a + step)
            seen = clen + b
            rows = q[a:b, h * group:(h + 1) * group].reshape(-1, d)
            p = torch.mm(rows, kt[:, :seen].contiguous()).mul_(1.0 / math.sqrt(d))
            p = p.view(b - a, group, seen)
            late = torch.arange(seen, device=DEV)[None] > (
                clen + torch.arange(a, b, device=DEV))[:, None]
            p.masked_fill_(late[:, None], -math.inf)
            p = p.sub_(p.amax(-1, keepdim=True)).exp_().view(-1, seen)
            o = torch.mm(p, vh[:seen]) / p.sum(-1, keepdim=True)
            out[a:b, h * group:(h + 1) * group] = o.view(b - a, group, d)
    return out


def exact(case, seed):
    outs, scales = [], ([], [])
    clen = case["clen"]
    for layer in range(case["layers"]):
        q, k, v = _tokens(case, seed, layer, "new")
        qf = q.double()
        if case["extra"] == "qk_norm":
            qg, kg = _gains(case, seed)
            # The path keeps the normalized rows in bf16, as the model does.
            qf = _rms(q, qg).to(torch.bfloat16)
            k = _rms(k, kg).to(torch.bfloat16)
        if case["extra"]:
            qf = _rope(qf, case, clen)
            k = _rope(k, case, clen).to(torch.bfloat16)
            if case["kind"] != "ingest":   # attention reads the rotated q in bf16
                qf = qf.to(torch.bfloat16).double()
        if case["kind"] == "ingest":
            k8, ks = _quantize(k)
            v8, vs = _quantize(v)
            outs.append(qf)
        else:
            if clen:
                ko, vo = _tokens(case, seed, layer, "old")
                k, v = torch.cat([ko, k]), torch.cat([vo, v])
            k8, ks = _quantize(k)
            v8, vs = _quantize(v)
            outs.append(_attend(qf, k8 * ks.double()[..., None], v8 * vs.double()[..., None],
                                case))
        scales[0].append(ks[-case["n"]:])
        scales[1].append(vs[-case["n"]:])
        del k8, v8
    out = outs[0] if case["kind"] == "ingest" else torch.stack(outs)
    if case["paged"]:   # the slabs' order is the block table's: the attention stands for them
        return {"out": out, "k": None, "v": None, "k_scale": None, "v_scale": None}
    return {"out": out, "k": None, "v": None, "k_scale": torch.stack(scales[0]).double(),
            "v_scale": torch.stack(scales[1]).double()}
