"""The workloads this package is measured on: decode attention over a paged latent cache at the sizes
a serving process meets, and the three kernels beside it (cache-row writer, prefill context gather,
decode query prep), each called through the package's public entry points.

    listed()            the named workloads
    draw(rng)           one more workload of the same ranges
    prepare(case, seed) inputs, caches and handles on the GPU
    run(state)          one pass; returns its outputs
    work(case)          bytes and flops a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the outputs in float64 torch

`kind` says which entry point a workload calls:
    mqa     `impl.forward_mqa`, the attention backend's decode, every layer of a step; `layers` > 0
            records that many layers (each with a cache of its own) into a HIP graph, as a serving
            engine does with its decode step, and a pass replays it; `layers` 0 is one eager call
    forward `qmla.forward`, query parts in, (output, lse) out
    fixed   `qmla.decode_attention_fwd`, the split-KV surface with its partials buffer
    write   `qmla.do_kv_cache_update`
    gather  `qmla.gather_cache`
    prep    `qmla.mla_decode_prep`
"""
import math
import os
import sys
from types import SimpleNamespace

import torch

if os.path.abspath("qwen-mla-vllm_amd") not in sys.path:
    sys.path.insert(0, os.path.abspath("qwen-mla-vllm_amd"))

import qmla  # noqa: E402
from qmla.backend import DecodeMetadataBuilder, QwenMLAHipImpl  # noqa: E402
from qmla.synth import lognormal_lens, make_case, uniform_lens  # noqa: E402


def _decode(name, kind, kv, rms, d_c, rope, heads, batch, page, dist, ctx, lo, hi, *, amp=1.0, qrows=1, groups=1,
            splits=0, layers=0, lens_seed=1):
    """dist: how the context lengths are spread: "fixed" (ctx each), "uniform" in [lo, hi] or
    "lognormal" with median ctx and sigma 0.5, clipped to [lo, hi]."""
    return dict(name=name, kind=kind, kv=kv, rms=rms, d_c=d_c, rope=rope, heads=heads, batch=batch, page=page,
                dist=dist, ctx=ctx, lo=lo, hi=hi, amp=amp, qrows=qrows, groups=groups, splits=splits, layers=layers,
                lens_seed=lens_seed)


def listed():
    return [
        # one user chatting: 16 layers' decode of a single short request in the engine's decode graph
        _decode("graph_fp8_b1", "mqa", "fp8", "log8", 512, 64, 24, 1, 64, "fixed", 1300, 1300, 1300, amp=4.0, layers=16),
        # a few requests on a bf16 cache in small pages, one eager layer: launch and host latency count
        _decode("bf16_b4", "mqa", "bf16", "bf16", 512, 64, 24, 4, 16, "fixed", 2048, 2048, 2048),
        # an ordinary chat batch in the decode graph: the deployed FP8 row (rank 768, packed rope 232)
        # in large pages, an odd number of requests, a few thousand tokens each, 4 layers
        _decode("graph_fp8_r768_b23", "mqa", "fp8", "log8", 768, 232, 24, 23, 784, "lognormal", 3000, 100, 16384,
                amp=4.0, layers=4),
        # the headline: FP8 with log8 codes, 128 long requests
        _decode("fp8_b128", "forward", "fp8", "log8", 512, 64, 24, 128, 64, "lognormal", 16384, 1024, 65536, amp=4.0,
                lens_seed=2),
        # long requests on a bf16 cache
        _decode("bf16_b64", "mqa", "bf16", "bf16", 512, 64, 24, 64, 64, "uniform", 0, 4096, 32768),
        # speculative verify: 4 query tokens a request, all heads on one latent row
        _decode("verify_fp8_b64x4", "mqa", "fp8", "log8", 512, 64, 24, 64, 64, "lognormal", 16384, 1024, 65536, amp=4.0,
                qrows=4, lens_seed=5),
        # speculative verify on the grouped latent (two groups of 256 columns)
        _decode("gla_fp8_b48x4", "forward", "fp8", "log8", 512, 64, 24, 48, 64, "uniform", 0, 8192, 32768, qrows=4,
                groups=2, lens_seed=4),
        # the wide latent at long context through the split-KV surface, 1600-token pages (the largest)
        _decode("wide_bf16_b32", "fixed", "bf16", "bf16", 1792, 64, 24, 32, 1600, "fixed", 65536, 65536, 65536,
                splits=16),
        # the deployed FP8 row at rank 1792, a mid-sized ragged batch
        _decode("fp8_r1792_b19", "mqa", "fp8", "log8", 1792, 232, 24, 19, 784, "lognormal", 8192, 500, 32768, amp=4.0,
                lens_seed=3),
        # a prefill chunk's rows into the FP8 cache: ragged prompts, pages in random order
        dict(name="write_fp8_n12001", kind="write", kv="fp8", rms="log8", d_c=512, rope=64, heads=24, n=12001, seqs=7,
             page=64),
        # chunked prefill: the cached context of a few prompts back into a dense bf16 buffer
        dict(name="gather_fp8_n20000", kind="gather", kv="fp8", rms="log8", d_c=512, rope=64, heads=24, n=20000, seqs=5,
             page=64),
        # the query prep of one layer's decode step
        dict(name="prep_b128", kind="prep", d_c=512, rope=64, heads=24, head_dim=256, kv_heads=4, declared=296, n=128),
    ]


# the cache rows that are deployed, and the page sizes they come in:
# (kv, rms, d_c, rope, heads, amp)
_ROWS = [
    ("fp8", "log8", 512, 64, 24, 4.0), ("fp8", "log8", 512, 64, 24, 4.0), ("fp8", "log8", 512, 64, 24, 1.0),
    ("bf16", "bf16", 512, 64, 24, 1.0), ("bf16", "bf16", 512, 64, 24, 1.0),
    ("fp8", "log8", 768, 232, 24, 4.0), ("fp8", "e4m3", 768, 232, 24, 1.0), ("fp8", "log8", 768, 116, 12, 4.0),
    ("fp8", "bf16", 512, 64, 24, 1.0), ("fp8", "e4m3", 512, 64, 24, 1.0),
    ("bf16", "bf16", 256, 116, 12, 1.0), ("bf16", "bf16", 768, 116, 12, 1.0),
    ("fp8", "log8", 1792, 232, 24, 4.0), ("bf16", "bf16", 1792, 64, 24, 1.0),
]
_DRAW_BYTES = 2.0e9      # cached bytes of a drawn decode at most
_DRAW_ROW_TOKENS = 5.0e6  # cached tokens x verify tokens at most


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 8 + ["write", "gather", "prep"])
    if kind in ("write", "gather"):
        kv, rms, d_c, rope, heads, _ = rng.choice(_ROWS)
        n = _log_int(rng, 16, 200_000 if d_c < 1000 else 60_000)
        return dict(kind=kind, kv=kv, rms=rms, d_c=d_c, rope=rope, heads=heads, n=n, seqs=rng.randint(1, min(n, 24)),
                    page=rng.choice([16, 64, 128, 784]))
    if kind == "prep":
        d_c = rng.choice([256, 512, 768])
        return dict(kind="prep", d_c=d_c, rope=64, heads=24, head_dim=256, kv_heads=4, declared=296,
                    n=_log_int(rng, 1, 512))
    kv, rms, d_c, rope, heads, amp = rng.choice(_ROWS)
    batch = _log_int(rng, 1, 160)
    ctx = _log_int(rng, 200, 32768)
    qrows, groups, splits, layers = 1, 1, 0, 0
    how = "mqa" if rms in ("log8", "bf16") and not (kv == "fp8" and rms == "bf16") else "forward"
    how = rng.choice([how, how, "forward", "fixed"])
    if how != "fixed" and d_c < 1000 and rng.random() < 0.3:
        qrows = rng.choice([2, 4])
    if how == "forward" and (kv, rms, d_c) == ("fp8", "log8", 512) and rng.random() < 0.5:
        groups = 2
    if how == "fixed":
        splits = rng.choice([4, 8, 16, 32])
    if how == "mqa" and qrows == 1 and batch <= 32 and ctx <= 4096 and rng.random() < 0.6:
        layers = rng.choice([2, 4, 8])
    esz = 1 if kv == "fp8" else 2
    per = ctx * 1.15 * max(1, layers)
    batch = max(1, min(batch, int(_DRAW_BYTES / (per * (d_c + rope + heads) * esz)), int(_DRAW_ROW_TOKENS / (per * qrows))))
    c = _decode("", how, kv, rms, d_c, rope, heads, batch, rng.choice([16, 64, 64, 128, 400, 784]),
                rng.choice(["lognormal", "lognormal", "uniform", "fixed"]), ctx, max(1, ctx // 8), 2 * ctx, amp=amp,
                qrows=qrows, groups=groups, splits=splits, layers=layers, lens_seed=rng.randint(1, 10 ** 6))
    del c["name"]
    return c


def _lens(c):
    if c["dist"] == "fixed":
        return [c["ctx"]] * c["batch"]
    if c["dist"] == "uniform":
        return uniform_lens(c["batch"], c["lo"], c["hi"], seed=c["lens_seed"])
    return lognormal_lens(c["batch"], c["ctx"], 0.5, c["lo"], c["hi"], seed=c["lens_seed"])


def _parts(n, seqs):
    """n tokens over `seqs` sequences, unevenly."""
    w = [1 + (i * 7) % 5 for i in range(seqs)]
    out = [max(1, n * x // sum(w)) for x in w]
    out[-1] += n - sum(out)
    while out[-1] < 1:                       # every sequence keeps a token
        k = max(range(seqs), key=lambda i: out[i])
        out[k] -= 1
        out[-1] += 1
    return out


def _mode(c):
    return "bf16_bytes" if c["kv"] == "fp8" and c["rms"] == "bf16" else c["rms"]


def _paged(c, seed):
    return make_case(batch=c["batch"], heads=c["heads"], d_c=c["d_c"], rope_w=c["rope"], page_size=c["page"],
                     lens=_lens(c), kv=c["kv"], rms_mode=_mode(c), seed=seed, device="cuda", qrows=c["qrows"],
                     groups=c["groups"], amp=c["amp"], q_amp=2.0, rms="row")


def _layer_seeds(c, seed):
    return [seed * 64 + k for k in range(max(1, c["layers"]))]


def _mqa_layer(c, case):
    """What the engine holds for one attention layer and step: the backend impl with its workspace,
    the absorbed query with its declared tail, vLLM's 3-D cache view and the step's metadata."""
    rows, heads, d_c, rope = case.q_nope.shape[0], c["heads"], c["d_c"], c["rope"]
    impl = QwenMLAHipImpl(kv_lora_rank=d_c, scale=case.sm_scale)
    impl.rms_offset, impl.mla_local_heads, impl.mla_kv_fp8 = d_c + rope, heads, c["kv"] == "fp8"
    impl.mla_packed_rope = rope
    q = torch.zeros(rows, heads, d_c + rope + heads + -(rope + heads) % 8, dtype=torch.bfloat16, device="cuda")
    q[..., :d_c] = case.q_nope
    q[..., d_c:d_c + rope] = case.q_pe
    n = rows // c["qrows"]
    table = case.block_table.view(n, c["qrows"], -1)[:, 0].contiguous()
    lens = case.seq_lens.view(n, c["qrows"])[:, -1].contiguous()
    md = DecodeMetadataBuilder(max_rows=rows).build_decode(table, lens, rows)
    impl.reserve_decode_workspace(rows, q.device, qrows=c["qrows"])
    meta = SimpleNamespace(causal=True, num_decode_tokens=rows, decode=md)
    return impl, q, case.cache[:, :, 0, :], meta, SimpleNamespace(_k_scale=case.k_scale)


def _write_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, d_c, rope, heads, page = c["n"], c["d_c"], c["rope"], c["heads"], c["page"]
    kv_c = (torch.randn(n, d_c, generator=g, device="cuda") * 2.0).to(torch.bfloat16)
    k_pe = torch.cat([torch.randn(n, rope, generator=g, device="cuda") * 2.0,
                      torch.exp(torch.randn(n, heads, generator=g, device="cuda") * 0.6)], -1).to(torch.bfloat16)
    lens = _parts(n, c["seqs"])
    pages = [-(-x // page) for x in lens]
    ids = torch.randperm(sum(pages) + 5, generator=torch.Generator().manual_seed(seed))
    slots, at = [], 0
    for x, p in zip(lens, pages):            # a sequence's tokens fill its pages in order
        t = torch.arange(x)
        slots.append(ids[at:at + p][t // page] * page + t % page)
        at += p
    per = 2 * heads if _mode(c) == "bf16_bytes" else heads
    row = -(-(d_c + rope + per) // 16) * 16
    dtype = torch.uint8 if c["kv"] == "fp8" else torch.bfloat16
    cache = torch.zeros(len(ids), page, row, dtype=dtype, device="cuda")
    scale = torch.tensor(2.0 * math.sqrt(2.0 * math.log(n * (d_c + rope))) / 448.0, device="cuda")
    return kv_c, k_pe, cache, torch.cat(slots).cuda(), scale


def _gather_inputs(c, seed):
    lens = _parts(c["n"], c["seqs"])
    case = make_case(batch=c["seqs"], heads=c["heads"], d_c=c["d_c"], rope_w=c["rope"], page_size=c["page"], lens=lens,
                     kv=c["kv"], rms_mode=_mode(c), seed=seed, device="cuda", rms="spread")
    t = torch.tensor(lens)
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), t.cumsum(0)]).to(torch.int32).cuda()
    seq = torch.repeat_interleave(torch.arange(c["seqs"], dtype=torch.int32), t).cuda()
    return case, cu, seq


def _prep_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, heads, hd, rd, d_c = c["n"], c["heads"], c["head_dim"], c["rope"], c["d_c"]

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    up = (rnd(heads * (hd - rd), d_c) * d_c ** -0.5).to(torch.bfloat16)
    table = qmla.partial_rope_table(range(rd // 2), rd, 1e7, 32768, device="cuda", dtype=torch.bfloat16)
    return dict(positions=torch.randint(0, 32768, (n,), generator=g, device="cuda"), q=rnd(n, heads, hd).to(torch.bfloat16),
                latent=rnd(n, d_c).to(torch.bfloat16), k_rope=rnd(n, c["kv_heads"] * rd).to(torch.bfloat16), k_up_raw=up,
                k_gain=qmla.k_gain((rnd(hd) * 0.1).to(torch.bfloat16), rd), cos_sin_cache=table)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "write":
        return c, _write_inputs(c, seed)
    if kind == "gather":
        paged, cu, seq = _gather_inputs(c, seed)
        return c, paged, cu, seq, torch.zeros(c["n"], paged.row, dtype=torch.bfloat16, device="cuda")
    if kind == "prep":
        return c, _prep_inputs(c, seed)
    paged = [_paged(c, s) for s in _layer_seeds(c, seed)]
    if kind == "forward":
        return c, paged[0], qmla.Workspace()
    if kind == "fixed":
        p, d_c, rope = paged[0], c["d_c"], c["rope"]
        rows, heads = p.q_nope.shape[:2]
        q = torch.cat([p.q_nope, p.q_pe], -1)
        o = torch.empty(rows, heads, d_c, dtype=torch.bfloat16, device="cuda")
        lse = torch.empty(rows, heads, dtype=torch.float32, device="cuda")
        logits = torch.empty(rows, heads, c["splits"], d_c + 1, dtype=torch.float32, device="cuda")
        return c, p, q, o, lse, logits
    layers = [_mqa_layer(c, p) for p in paged]
    if not c["layers"]:
        return c, layers, None, None
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):            # one eager step first, as engines warm up before they capture
        for impl, *args in layers:
            impl.forward_mqa(*args)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [impl.forward_mqa(*args)[0] for impl, *args in layers]
    return c, layers, graph, outs


def run(state):
    c, kind = state[0], state[0]["kind"]
    if kind == "mqa":
        _, layers, graph, outs = state
        if graph is not None:
            graph.replay()
            return outs
        impl, *args = layers[0]
        return impl.forward_mqa(*args)[0]
    if kind == "forward":
        _, p, ws = state
        return qmla.forward(p.q_nope, p.q_pe, p.cache, p.block_table, p.seq_lens, page_size=p.page_size,
                            sm_scale=p.sm_scale, fp8_rms=c["rms"] if c["kv"] == "fp8" else "log8", k_scale=p.k_scale,
                            qrows=p.qrows, groups=p.groups, workspace=ws)
    if kind == "fixed":
        _, p, q, o, lse, logits = state
        qmla.decode_attention_fwd(q, p.cache, p.cache[..., :c["d_c"]], o, lse, p.block_table, p.seq_lens, logits,
                                  c["splits"], p.sm_scale, p.page_size, k_scale=p.k_scale, is_mla=True,
                                  rms_offset=p.rms_offset, rms_bf16=c["kv"] == "fp8" and c["rms"] == "bf16",
                                  rms_log8=c["rms"] == "log8")
        return o, lse
    if kind == "write":
        kv_c, k_pe, cache, slots, scale = state[1]
        qmla.do_kv_cache_update(kv_c, k_pe, cache, slots, "fp8" if c["kv"] == "fp8" else "auto", scale,
                                packed_rope=c["rope"], n_heads=c["heads"], rms_mode=c["rms"])
        return cache
    if kind == "gather":
        _, p, cu, seq, dst = state
        fp8 = c["kv"] == "fp8"
        qmla.gather_cache(src_cache=p.cache[:, :, 0, :], dst=dst, block_table=p.block_table, cu_seq_lens=cu,
                          token_to_seq=seq, num_tokens=c["n"], kv_cache_dtype="fp8" if fp8 else "auto", scale=p.k_scale,
                          mla_rms=(p.rms_offset, c["heads"], c["rms"]) if fp8 else None)
        return dst
    return qmla.mla_decode_prep(**state[1], **_prep_args(c))


def _prep_args(c):
    return dict(head_offset=0, rope_group=c["heads"] // c["kv_heads"], rope_first=0, rope_span=c["kv_heads"],
                declared_rope=c["declared"], eps=1e-6)


def work(case):
    c, kind = case, case["kind"]
    if kind == "prep":
        n, heads, hd, rd, d_c = c["n"], c["heads"], c["head_dim"], c["rope"], c["d_c"]
        nope = hd - rd
        by = 2 * (n * (heads * hd + d_c + c["kv_heads"] * rd) + heads * nope * d_c + n * rd + n * c["declared"]
                  + n * heads * (nope + c["declared"])) + 4 * rd + 8 * n
        return {"bytes": by, "flops": 2 * n * heads * nope * d_c}
    d_c, rope, heads = c["d_c"], c["rope"], c["heads"]
    esz = 1 if c["kv"] == "fp8" else 2
    per = (d_c + rope) * esz + heads * (1 if c["rms"] in ("log8", "e4m3") else 2)   # cached bytes of one token
    if kind in ("write", "gather"):
        dense = 2 * (d_c + rope + heads)
        return {"bytes": c["n"] * (per + dense + (8 if kind == "write" else 4)), "flops": c["n"] * (d_c + rope + heads)}
    lens, qr, groups = _lens(c), c["qrows"], c["groups"]
    rows, dv = c["batch"] * qr, d_c // groups
    pages = sum(-(-x // c["page"]) for x in lens)
    by = sum(lens) * per + rows * heads * (2 * (dv + rope) + 2 * dv + 4) + 4 * (pages + rows)
    seen = sum(max(0, x - j) for x in lens for j in range(qr))
    return {"bytes": by * max(1, c["layers"]), "flops": 2 * seen * heads * (2 * dv + rope) * max(1, c["layers"])}


def tolerance(case):
    if case["kind"] in ("write", "gather"):
        return "exact"                       # one rounding of each value, stated by the cache format
    # bf16 outputs measure 1.7e-3 to 1.9e-3 off float64 (their own rounding is most of it); the prep's
    # rotation rounds every bf16 product and sum and measures 2.7e-3
    return {"rel": 1.2e-2 if case["kind"] == "prep" else 8e-3}


def _latent_rows(case, idx):
    """The cached rows `idx` as float64: values [n, d_c + rope] and the divisors [n, heads]."""
    w, h = case.d_c + case.rope_w, case.heads
    row = case.cache.view(-1, case.row)[idx]
    if case.kv == "bf16":
        return row[:, :w].double(), row[:, w:w + h].double()
    scale = case.k_scale.double()
    val = row[:, :w].view(torch.float8_e4m3fn).double() * scale
    if case.rms_mode == "log8":
        return val, torch.exp2(-3.0 + row[:, w:w + h].double() * (6.0 / 255.0))
    if case.rms_mode == "e4m3":
        return val, row[:, w:w + h].contiguous().view(torch.float8_e4m3fn).double() * scale
    return val, row[:, w:w + 2 * h].contiguous().view(torch.bfloat16).double()


def _exact_decode(case):
    """Attention of every query row over its cached tokens, in float64."""
    rows, h = case.q_nope.shape[:2]
    dv, hg = case.d_c // case.groups, h // case.groups
    out = torch.zeros(rows, h, dv, dtype=torch.float64, device="cuda")
    lse = torch.full((rows, h), float("-inf"), dtype=torch.float64, device="cuda")
    lens = case.seq_lens.tolist()
    for b in range(0, rows, case.qrows):
        n = lens[b + case.qrows - 1]
        t = torch.arange(n, device="cuda")
        page = case.block_table[b + case.qrows - 1].long()[t // case.page_size]
        val, rms = _latent_rows(case, page * case.page_size + t % case.page_size)
        rms = torch.where(rms > 0, rms, torch.ones_like(rms)).t()
        lat, pe = val[:, :case.d_c], val[:, case.d_c:]
        for r in range(b, b + case.qrows):
            for g in range(case.groups):
                hs = slice(g * hg, (g + 1) * hg)
                v = lat[:, g * dv:(g + 1) * dv]
                s = (case.q_nope[r, hs].double() @ v.t() + case.q_pe[r, hs].double() @ pe.t()) / rms[hs] * case.sm_scale
                s = s[:, :lens[r]]
                if lens[r] > 0:
                    lse[r, hs] = torch.logsumexp(s, -1)
                    out[r, hs] = torch.softmax(s, -1) @ v[:lens[r]]
    return out, lse


def _exact_prep(c, a):
    n, heads, hd, rd = c["n"], c["heads"], c["head_dim"], c["rope"]
    nope, group = hd - rd, heads // c["kv_heads"]
    trig = a["cos_sin_cache"].double()[a["positions"]]
    cos, sin = trig[:, None, :rd // 2], trig[:, None, rd // 2:]

    def rotate(x):
        x1, x2 = x[..., :rd // 2], x[..., rd // 2:]
        return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], -1)

    key = a["k_rope"].double().view(n, c["kv_heads"], rd)
    up = (a["latent"].double() @ a["k_up_raw"].double().t()).view(n, heads, nope)
    squares = up.square().sum(-1) + key.square().sum(-1).repeat_interleave(group, 1)
    rms = (squares / hd + 1e-6).sqrt()
    q_out = torch.zeros(n, heads, nope + c["declared"], dtype=torch.float64, device="cuda")
    q_out[..., :nope] = a["q"][..., rd:].double()
    turned = rotate(a["q"][..., :rd].double())
    for h in range(heads):
        at = nope + (h // group) * rd
        q_out[:, h, at:at + rd] = turned[:, h]
    k_pe = torch.zeros(n, c["declared"], dtype=torch.float64, device="cuda")
    k_pe[:, :c["kv_heads"] * rd] = rotate(key * a["k_gain"].double()).reshape(n, -1)
    k_pe[:, c["kv_heads"] * rd:c["kv_heads"] * rd + heads] = rms
    return q_out, k_pe


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "write":
        if c["kv"] == "fp8":
            return None                      # bytes
        kv_c, k_pe, cache, slots, _ = _write_inputs(c, seed)
        want = torch.zeros(cache.numel() // cache.shape[-1], cache.shape[-1], dtype=torch.float64, device="cuda")
        want[slots, :c["d_c"] + k_pe.shape[-1]] = torch.cat([kv_c, k_pe], -1).double()
        return want.view(cache.shape)
    if kind == "gather":
        paged, _, _ = _gather_inputs(c, seed)
        want, at = torch.zeros(c["n"], paged.row, dtype=torch.float64, device="cuda"), 0
        for b, x in enumerate(_parts(c["n"], c["seqs"])):
            t = torch.arange(x, device="cuda")
            idx = paged.block_table[b].long()[t // c["page"]] * c["page"] + t % c["page"]
            val, rms = _latent_rows(paged, idx)
            w = val.shape[1]
            want[at:at + x, :w], want[at:at + x, w:w + c["heads"]] = val, rms
            at += x
        return want
    if kind == "prep":
        return _exact_prep(c, _prep_inputs(c, seed))
    outs = [_exact_decode(_paged(c, s)) for s in _layer_seeds(c, seed)]
    if kind == "mqa":
        return [o for o, _ in outs] if c["layers"] else outs[0][0]
    return outs[0]
