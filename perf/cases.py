"""The work that a serving engine has this library do for one layer, as cases that can be timed.

Five kinds of call, each through the entry point that an engine uses:

* ``decode``: absorbed-MLA paged decode of one layer over a planned batch (``lib.mla_decode``);
* ``prefill``: chunked causal prefill over per-head K/V pages (``lib.mla_prefill``);
* ``backend_prefill``: the attention backend's prefill over the latent pool (store of the chunk, gather,
  decompression, attention; ``MLAAttnBackend.forward``);
* ``layer_decode`` / ``layer_prefill``: a whole MLA layer (projections, norms, RoPE, attention,
  output projection; ``MLAAttentionLayer.forward``), decode steps also replayed from a HIP graph that
  was captured through the backend's capture hooks, as an engine runs them.

Lengths are drawn from the case's own ``lens_seed``, so a case's work does not depend on the seed of
its values; page tables, queries, keys and weights come from the seed. Values are N(0, 1) in bf16, weights
N(0, 1 / fan_in).
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-sglang_amd"))

from minisgl_amd.attention import create_attention_backend  # noqa: E402
from minisgl_amd.config import MLAConfig  # noqa: E402
from minisgl_amd.core import Batch, Context, Req, reset_global_ctx, set_global_ctx  # noqa: E402
from minisgl_amd.kernel import lib  # noqa: E402
from minisgl_amd.kvcache import create_kvcache_pool  # noqa: E402
from minisgl_amd.layers import MLAAttentionLayer, MLALayerConfig, MLAWeights, softmax_mscale  # noqa: E402

SCALE = 192 ** -0.5
YARN = (("rope_type", "yarn"), ("factor", 32.0), ("original_max_position_embeddings", 4096), ("beta_fast", 1.0),
        ("beta_slow", 1.0), ("mscale", 1.0), ("mscale_all_dim", 1.0))
HIDDEN, Q_LORA, MAX_POS, ROPE_THETA, EPS = 7168, 1536, 32768, 50000.0, 1e-6


def listed():
    return [
        # one user's chat, some 1,500 tokens in: the smallest decode call, latency and launches
        dict(name="decode-single", kind="decode", batch=1, heads=64, page=64, lo=1400, hi=1600, lens_seed=1),
        # the Kimi-K2 shape of the benchmark: 64 requests of 1k to 8k tokens
        dict(name="decode-batch", kind="decode", batch=64, heads=64, page=64, lo=1024, hi=8192, lens_seed=0),
        # the engine's default page size, a medium batch of an odd size
        dict(name="decode-page1", kind="decode", batch=19, heads=64, page=1, lo=300, hi=4000, lens_seed=2),
        # long documents: few requests of 32k to 128k tokens
        dict(name="decode-long", kind="decode", batch=8, heads=64, page=64, lo=32768, hi=131072, lens_seed=0),
        # one of eight tensor-parallel ranks of a 64-head model
        dict(name="decode-heads8", kind="decode", batch=64, heads=8, page=64, lo=1024, hi=8192, lens_seed=3),
        # a 16-head rank and short contexts at page size 1 (the CPU reference workload's shape)
        dict(name="decode-heads16-short", kind="decode", batch=4, heads=16, page=1, lo=64, hi=512, lens_seed=4),
        # 128 heads on one GPU (data-parallel attention)
        dict(name="decode-heads128", kind="decode", batch=32, heads=128, page=64, lo=1024, hi=8192, lens_seed=5),
        # short ragged prompts and continuations over per-head pages
        dict(name="prefill-ragged", kind="prefill", batch=6, heads=64, page=64, elo=1, ehi=300, plo=0, phi=1000,
             lens_seed=6),
        # the benchmark's chunked prefill: four chunks of 2048 on prefixes of up to 8k
        dict(name="prefill-chunk", kind="prefill", batch=4, heads=64, page=64, elo=2048, ehi=2048, plo=0, phi=8192,
             lens_seed=0),
        # a rank's prefill from the latent pool at the default page size, medium chunks
        dict(name="backend-prefill", kind="backend_prefill", batch=3, heads=64, page=1, elo=200, ehi=1000, plo=0,
             phi=3000, lens_seed=7),
        # a decode step of a whole layer, replayed from a graph
        dict(name="layer-decode", kind="layer_decode", batch=64, heads=64, page=64, lo=1024, hi=8192, lens_seed=0,
             graph=True),
        # a prompt chunk through a whole layer
        dict(name="layer-prefill", kind="layer_prefill", batch=2, heads=64, page=64, elo=500, ehi=1100, plo=0, phi=2048,
             lens_seed=8),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["prefill", "prefill", "backend_prefill", "layer_decode", "layer_decode",
                                        "layer_prefill"])
    case = dict(kind=kind, lens_seed=rng.randrange(1 << 30))
    if kind == "decode":
        case["heads"] = rng.choice([8, 8, 16, 32, 64, 64, 64, 128, rng.randint(1, 128)])
        case["page"] = rng.choice([1, 1, 16, 64, 64, 64, 128])
        case["batch"] = _log(rng, 1, 128)
        # at most the tokens of the longest listed batch, a request at most 128k; 128 heads read them twice
        most = min(131072, 650000 // case["batch"] // (1 if case["heads"] <= 64 else 2))
        case["hi"] = _log(rng, 64, most)
        case["lo"] = rng.randint(max(1, case["hi"] // 8), case["hi"])
    elif kind == "layer_decode":
        case["heads"] = rng.choice([8, 16, 64, 64])
        case["page"] = rng.choice([1, 64, 64])
        case["batch"] = _log(rng, 1, 64)
        case["hi"] = _log(rng, 64, min(MAX_POS, 360000 // case["batch"]))
        case["lo"] = rng.randint(max(1, case["hi"] // 8), case["hi"])
        case["graph"] = rng.random() < 0.75
    else:
        case["heads"] = rng.choice([8, 16, 64, 64])
        case["page"] = rng.choice([64, 64, 128]) if kind == "prefill" else rng.choice([1, 64])
        case["batch"] = _log(rng, 1, 16)
        case["ehi"] = _log(rng, 8, max(8, (8192 if kind == "prefill" else 3000) // case["batch"]))
        case["elo"] = rng.randint(max(1, case["ehi"] // 4), case["ehi"])
        case["phi"] = rng.choice([0, _log(rng, 64, min(8192, (16000 if kind == "prefill" else 6000) // case["batch"]))])
        case["plo"] = rng.randint(0, case["phi"])
        while case["phi"] and work(case)["flops"] > 2.5e12:  # no more than the largest listed batch
            case["phi"] //= 2
            case["plo"] = min(case["plo"], case["phi"])
    return case


# ---------------------------------------------------------------------------------------- sizes


def _lens(case):
    r = random.Random(case["lens_seed"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]


def _chunks(case):
    """Extends and prefixes of a prefill batch."""
    r = random.Random(case["lens_seed"])
    ext = [r.randint(case["elo"], case["ehi"]) for _ in range(case["batch"])]
    return ext, [r.randint(case["plo"], case["phi"]) for _ in range(case["batch"])]


def _weight_params(heads):
    return (Q_LORA + 576) * HIDDEN + heads * 192 * Q_LORA + heads * 256 * 512 + HIDDEN * heads * 128


def work(case):
    """Each input read once and each output written once, and the products that the path needs."""
    H, page, kind = case["heads"], case["page"], case["kind"]
    if kind in ("decode", "layer_decode"):
        lens = _lens(case)
        B, T = len(lens), sum(lens)
        attn_flops = 2 * T * H * (576 + 512)
        table = sum(-(-n // page) for n in lens) * 4 + 4 * B
        if kind == "decode":
            return {"bytes": T * 1152 + table + B * H * (576 + 512) * 2 + B * H * 4, "flops": attn_flops}
        return {"bytes": _weight_params(H) * 2 + T * 1152 + table + 2 * B * HIDDEN * 2,
                "flops": attn_flops + 2 * B * _weight_params(H)}
    ext, pre = _chunks(case)
    T, keys = sum(ext), sum(ext) + sum(pre)
    pairs = sum(e * p + e * (e + 1) // 2 for e, p in zip(ext, pre))
    attn_flops = pairs * H * 2 * (192 + 128)
    table = sum(-(-(e + p) // page) for e, p in zip(ext, pre)) * 4
    if kind == "prefill":
        return {"bytes": (keys + T) * H * (192 + 128) * 2 + T * H * 4 + table, "flops": attn_flops}
    decompress = keys * H * 256 * 512 * 2
    if kind == "backend_prefill":
        return {"bytes": keys * 1152 + T * 1152 + H * 256 * 512 * 2 + T * H * (192 + 128) * 2 + T * H * 4 + table,
                "flops": attn_flops + decompress}
    proj = (Q_LORA + 576) * HIDDEN + H * 192 * Q_LORA + HIDDEN * H * 128
    return {"bytes": _weight_params(H) * 2 + keys * 1152 + 2 * T * HIDDEN * 2 + table,
            "flops": attn_flops + decompress + 2 * T * proj}


def tolerance(case):
    """bf16 results of fp32 sums: the attention's relative error is about 2e-3 (one rounding of the
    probabilities and of the output), a whole layer's about 6e-3 (five products with bf16 between them)."""
    return {"rel": 2.5e-2} if case["kind"].startswith("layer") else {"rel": 1e-2}


# --------------------------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(shape, gen, scale=1.0):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)
    return x if scale == 1.0 else x.mul_(scale)


def _pages(lens, page, gen):
    """Page ids of every request (a random permutation of the pool's pages) and the pool's page count."""
    need = [-(-n // page) for n in lens]
    num = sum(need) + 1
    perm = torch.randperm(num, generator=gen, device="cuda").to(torch.int32)
    rows, off = torch.zeros((len(lens), max(need)), dtype=torch.int32, device="cuda"), 0
    for b, n in enumerate(need):
        rows[b, :n] = perm[off : off + n]
        off += n
    return rows, num


def _prepare_decode(case, seed):
    gen, lens = _gen(seed), _lens(case)
    B, H = len(lens), case["heads"]
    pt, num = _pages(lens, case["page"], gen)
    ctas = lib.device_cu_count(torch.cuda.current_device())
    plan, slots = lib.decode_plan(lens, case["page"], ctas)
    ws_o, ws_lse = lib.decode_workspace(slots, H, "cuda")
    return dict(case=case, lens=lens, pt=pt, seq_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"),
                plan=torch.from_numpy(plan).cuda(), ctas=ctas, ws_o=ws_o, ws_lse=ws_lse,
                q=_randn((B, H, 576), gen), kv=_randn((num, case["page"], 576), gen),
                out=torch.empty((B, H, 512), dtype=torch.bfloat16, device="cuda"),
                lse=torch.empty((B, H), dtype=torch.float32, device="cuda"))


def _prepare_prefill(case, seed):
    gen = _gen(seed)
    ext, pre = _chunks(case)
    lens, H, T = [e + p for e, p in zip(ext, pre)], case["heads"], sum(ext)
    pt, num = _pages(lens, case["page"], gen)
    cu = torch.tensor([0] + ext).cumsum(0).to(torch.int32).cuda()
    return dict(case=case, ext=ext, lens=lens, pt=pt, cu=cu,
                seq_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"), q=_randn((T, H, 192), gen),
                k=_randn((num, case["page"], H, 192), gen), v=_randn((num, case["page"], H, 128), gen),
                out=torch.empty((T, H, 128), dtype=torch.bfloat16, device="cuda"),
                lse=torch.empty((T, H), dtype=torch.float32, device="cuda"))


def _engine(case, lens, ext, attn, gen):
    """Context, latent pool, backend and one batch, as an engine holds them. The requests' last ``ext``
    tokens are the step's new ones."""
    page = case["page"]
    pt, num = _pages(lens, page, gen)
    width = -(-pt.shape[1] * page // 32) * 32
    tokens = torch.zeros((len(lens) + 1, width), dtype=torch.int32, device="cuda")
    tokens[: len(lens), : pt.shape[1] * page] = (
        pt[:, :, None] * page + torch.arange(page, dtype=torch.int32, device="cuda")).flatten(1)
    reset_global_ctx()
    ctx = Context(page_size=page)
    set_global_ctx(ctx)
    ctx.page_table = tokens
    ctx.kv_cache = pool = create_kvcache_pool(attn, num, page, torch.bfloat16, torch.device("cuda"))
    pool.latent_cache(0).copy_(_randn(pool.latent_cache(0).shape, gen))
    ctx.attn_backend = backend = create_attention_backend("mla", attn)
    reqs = [Req(table_idx=b, cached_len=n - e, device_len=n) for b, (n, e) in enumerate(zip(lens, ext))]
    batch = Batch(reqs=reqs, phase="decode" if case["kind"] == "layer_decode" else "prefill")
    batch.padded_reqs = reqs
    batch.positions = torch.cat([torch.arange(r.cached_len, r.device_len) for r in reqs]).to(torch.int32).cuda()
    batch.out_loc = torch.cat([tokens[r.table_idx, r.cached_len : r.device_len] for r in reqs])
    return dict(case=case, lens=lens, ext=ext, ctx=ctx, pool=pool, backend=backend, batch=batch, tokens=tokens)


def _prepare_backend_prefill(case, seed):
    gen = _gen(seed)
    ext, pre = _chunks(case)
    H, T = case["heads"], sum(ext)
    s = _engine(case, [e + p for e, p in zip(ext, pre)], ext, MLAConfig(num_heads=H), gen)
    s["kv_b"] = _randn((H * 256, 512), gen, 512 ** -0.5)
    s["backend"].register_kv_b(0, s["kv_b"])
    s["backend"].prepare_metadata(s["batch"])
    s["q"], s["k_new"] = _randn((T, H, 192), gen), _randn((T, 576), gen)
    return s


def _weights(heads, gen):
    def lin(out_f, in_f):
        return _randn((out_f, in_f), gen, in_f ** -0.5)

    def norm(n):
        return (1.0 + 0.1 * torch.randn((n,), generator=gen, device="cuda")).to(torch.bfloat16)

    return MLAWeights(q_a=lin(Q_LORA, HIDDEN), q_a_norm=norm(Q_LORA), q_b=lin(heads * 192, Q_LORA),
                      kv_a=lin(576, HIDDEN), kv_a_norm=norm(512), kv_b=lin(heads * 256, 512),
                      o=lin(HIDDEN, heads * 128))


def _prepare_layer(case, seed):
    gen, H = _gen(seed), case["heads"]
    if case["kind"] == "layer_decode":
        lens = _lens(case)
        ext = [1] * len(lens)
    else:
        ext, pre = _chunks(case)
        lens = [e + p for e, p in zip(ext, pre)]
    attn = MLAConfig(num_heads=H, softmax_mscale=softmax_mscale(YARN))
    cfg = MLALayerConfig(attn=attn, hidden_size=HIDDEN, q_lora_rank=Q_LORA, rope_theta=ROPE_THETA,
                         max_position=MAX_POS, rms_eps=EPS, rope_scaling=YARN)
    s = _engine(case, lens, ext, attn, gen)
    s["weights"] = _weights(H, gen)
    s["layer"] = MLAAttentionLayer(0, cfg, s["weights"])
    s["x"] = _randn((sum(ext), HIDDEN), gen)
    backend, batch, ctx = s["backend"], s["batch"], s["ctx"]
    if not case.get("graph"):
        backend.prepare_metadata(batch)
        return s
    backend.init_capture_graph(max(lens), [len(lens)])
    backend.prepare_for_capture(batch)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream), ctx.forward_batch(batch):
        s["layer"].forward(s["x"])
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]), ctx.forward_batch(batch):
        s["y"] = s["layer"].forward(s["x"])
    s["lse"] = backend.last_lse
    backend.prepare_metadata(batch)
    backend.prepare_for_replay(batch)
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _prepare_decode(case, seed)
    if kind == "prefill":
        return _prepare_prefill(case, seed)
    if kind == "backend_prefill":
        return _prepare_backend_prefill(case, seed)
    return _prepare_layer(case, seed)


def run(state):
    s = state
    kind = s["case"]["kind"]
    if kind == "decode":
        lib.mla_decode(s["q"], s["kv"], s["pt"], s["seq_lens"], s["plan"], s["ctas"], s["ws_o"], s["ws_lse"], SCALE,
                       s["out"], s["lse"])
        return s["out"], s["lse"]
    if kind == "prefill":
        lib.mla_prefill(s["q"], s["k"], s["v"], s["pt"], s["cu"], s["seq_lens"], SCALE, s["out"], s["lse"])
        return s["out"], s["lse"]
    if "graph" in s:
        s["graph"].replay()
        return s["y"], s["lse"], s["pool"].latent_cache(0)
    reset_global_ctx()  # several engines' states can be alive here; a program has one
    set_global_ctx(s["ctx"])
    with s["ctx"].forward_batch(s["batch"]):
        if kind == "backend_prefill":
            y = s["backend"].forward(s["q"], s["k_new"], None, 0, s["batch"])
        else:
            y = s["layer"].forward(s["x"])
    return y, s["backend"].last_lse, s["pool"].latent_cache(0)


# ------------------------------------------------------------------------------- 64-bit results


def _attend(q, k, v, scale, first):
    """``q [n, H, d]``, ``k [H, L, d]``, ``v [H, L, e]``: row i sees keys up to ``first + i``."""
    n, H, _ = q.shape
    L = k.shape[1]
    out = torch.empty((n, H, v.shape[2]), dtype=torch.float64, device=q.device)
    lse = torch.empty((n, H), dtype=torch.float64, device=q.device)
    step = max(1, (1 << 26) // L)
    for h in range(H):
        for i in range(0, n, step):
            s = (q[i : i + step, h].contiguous() @ k[h].t()) * scale
            last = first + torch.arange(i, min(n, i + step), device=q.device)
            s.masked_fill_(torch.arange(L, device=q.device)[None] > last[:, None], -math.inf)
            m = s.amax(1, keepdim=True)
            p = (s - m).exp_()
            t = p.sum(1, keepdim=True)
            out[i : i + step, h] = (p @ v[h]) / t
            lse[i : i + step, h] = (m + t.log())[:, 0]
    return out, lse


def _attend_latent(q, rows, scale):
    """One request's absorbed decode: ``q [H, 576]`` over latent rows ``[L, 576]``."""
    s = (q @ rows.t()) * scale
    m = s.amax(1, keepdim=True)
    p = (s - m).exp_()
    t = p.sum(1, keepdim=True)
    return (p @ rows[:, :512]) / t, (m + t.log())[:, 0]


def _rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def _rope(x, pos):
    """Interleaved pairs of the last 64 dims rotated with YaRN's frequencies; x [n, ..., 64] in 64 bits."""
    base = 1.0 / ROPE_THETA ** (torch.arange(0, 64, 2, dtype=torch.float64, device=x.device) / 64)
    rs = dict(YARN)

    def dim_of(turns):
        return 64 * math.log(rs["original_max_position_embeddings"] / (turns * 2 * math.pi)) / (2 * math.log(ROPE_THETA))

    lo, hi = max(math.floor(dim_of(rs["beta_fast"])), 0), min(math.ceil(dim_of(rs["beta_slow"])), 31)
    ramp = ((torch.arange(32, dtype=torch.float64, device=x.device) - lo) / max(hi - lo, 1)).clamp(0.0, 1.0)
    a = pos.double()[:, None] * (base * (1 - ramp) + base / rs["factor"] * ramp)
    c, s = (t.reshape((len(pos),) + (1,) * (x.dim() - 2) + (32,)) for t in (a.cos(), a.sin()))
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack((e * c - o * s, o * c + e * s), -1).flatten(-2)


def _exact_latent_prefill(q, pool, tokens, lens, ext, kv_b, scale):
    """Prefill attention over the pool's rows, whose keys and values are decompressed per head."""
    H = q.shape[1]
    outs, lses, off = [], [], 0
    w = kv_b.double().view(H, 256, 512)
    for b, (n, e) in enumerate(zip(lens, ext)):
        rows = pool[tokens[b, :n].long()].double()
        k = torch.stack([torch.cat((rows[:, :512] @ w[h, :128].t(), rows[:, 512:]), 1) for h in range(H)])
        v = torch.stack([rows[:, :512] @ w[h, 128:].t() for h in range(H)])
        o, l = _attend(q[off : off + e], k, v, scale, n - e)
        outs.append(o)
        lses.append(l)
        off += e
    return torch.cat(outs), torch.cat(lses)


def exact(case, seed):
    s, kind, H = prepare(case, seed), case["kind"], case["heads"]
    page = case["page"]
    if kind == "decode":
        flat, outs = s["kv"].view(-1, 576), []
        for b, n in enumerate(s["lens"]):
            t = torch.arange(n, device="cuda")
            rows = flat[s["pt"][b, t // page].long() * page + t % page].double()
            outs.append(_attend_latent(s["q"][b].double(), rows, SCALE))
        return torch.stack([o for o, _ in outs]), torch.stack([l for _, l in outs])
    if kind == "prefill":
        outs, off = [], 0
        for b, (n, e) in enumerate(zip(s["lens"], s["ext"])):
            t = torch.arange(n, device="cuda")
            rows = s["pt"][b, t // page].long() * page + t % page
            k, v = (s[x].view(-1, H, s[x].shape[-1])[rows].transpose(0, 1).double().contiguous() for x in ("k", "v"))
            outs.append(_attend(s["q"][off : off + e].double(), k, v, SCALE, n - e))
            off += e
        return torch.cat([o for o, _ in outs]), torch.cat([l for _, l in outs])
    pool = s["pool"].latent_cache(0).view(-1, 576).clone()
    loc = s["batch"].out_loc.long()
    if kind == "backend_prefill":
        pool[loc] = s["k_new"]
        o, l = _exact_latent_prefill(s["q"].double(), pool, s["tokens"], s["lens"], s["ext"], s["kv_b"], SCALE)
        return o, l, None
    w, x, pos = s["weights"], s["x"].double(), s["batch"].positions
    scale = SCALE * softmax_mscale_of_yarn() ** 2
    q = (_rms(x @ w.q_a.double().t(), w.q_a_norm) @ w.q_b.double().t()).view(-1, H, 192)
    q = torch.cat((q[..., :128], _rope(q[..., 128:], pos)), -1)
    kv = x @ w.kv_a.double().t()
    new = torch.cat((_rms(kv[:, :512], w.kv_a_norm), _rope(kv[:, 512:], pos)), -1)
    pool = pool.double()
    pool[loc] = new
    if kind == "layer_prefill":
        o, l = _exact_latent_prefill(q, pool, s["tokens"], s["lens"], s["ext"], w.kv_b, scale)
    else:
        kv_b, outs = w.kv_b.double().view(H, 256, 512), []
        for b, n in enumerate(s["lens"]):
            q_lat = torch.stack([q[b, h, :128] @ kv_b[h, :128] for h in range(H)])
            o, l = _attend_latent(torch.cat((q_lat, q[b, :, 128:]), 1), pool[s["tokens"][b, :n].long()], scale)
            outs.append((torch.stack([kv_b[h, 128:] @ o[h] for h in range(H)]), l))
        o, l = torch.stack([o for o, _ in outs]), torch.stack([l for _, l in outs])
    return o.flatten(1) @ w.o.double().t(), l, None


def softmax_mscale_of_yarn():
    rs = dict(YARN)
    return 0.1 * rs["mscale_all_dim"] * math.log(rs["factor"]) + 1.0
