"""Performance cases of the paged-attention path: the calls an engine makes once per layer and scheduler step.

``listed()`` names the cases, ``draw()`` makes further ones over the same ranges.  Every case goes through the
package's public entry points: ``qwen3_attention_core`` (q/k norm + RoPE + KV store + attention, a Qwen3 layer's
whole step between its projections), ``attention`` (KV store + attention, any head size) or, for the options that
the layer seam does not carry (soft cap, quantized pages), the store followed by the kernel entry.

A case is a dict of plain values:

  step        "prefill", "decode" or "mixed" (decode sequences first, then prefill sequences, one call)
  entry       "core", "attention" or "kernel", as above
  heads, kv_heads, head_dim, page_size
  pages       "bf16", "fp8" (e4m3 codes, stored by the quantising store) or "int8" (codes the caller already has;
              the library has no writer for them, so such a case is the kernel entry alone)
  seqs, new_lo, new_hi, prefix_lo, prefix_hi    prefill sequences: new tokens and cached tokens before them
  shared      the cached tokens are one common document whose whole pages the sequences share
  decodes, ctx_lo, ctx_hi                       decode sequences: context lengths, the new token included
  soft_cap    0 = off
  lens        seeds the lengths, which are part of the case; the values and the page placement come from the seed
"""
import importlib.util
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """``vllm-jax_amd/`` under its module name (the folder's hyphen needs an import by path)."""
    if "vllm_jax_amd" not in sys.modules:
        path = os.path.join(ROOT, "vllm-jax_amd")
        spec = importlib.util.spec_from_file_location("vllm_jax_amd", os.path.join(path, "__init__.py"),
                                                      submodule_search_locations=[path])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["vllm_jax_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["vllm_jax_amd"]


pa = _package()

EPS, ROPE_THETA = 1e-6, 1e6


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _case(step, entry, heads, kv_heads, page_size, *, head_dim=128, pages="bf16", seqs=0, new=(0, 0), prefix=(0, 0),
          shared=False, decodes=0, ctx=(0, 0), soft_cap=0.0, lens=0, name=None):
    c = dict(step=step, entry=entry, heads=heads, kv_heads=kv_heads, head_dim=head_dim, page_size=page_size,
             pages=pages, seqs=seqs, new_lo=new[0], new_hi=new[1], prefix_lo=prefix[0], prefix_hi=prefix[1],
             shared=shared, decodes=decodes, ctx_lo=ctx[0], ctx_hi=ctx[1], soft_cap=float(soft_cap), lens=lens)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest step: four sequences of a short chat over 16-token pages (Qwen3-0.6B heads, the engine's
        # own smoke configuration).  Every layer of every generated token makes this call: latency and launches.
        _case("decode", "core", 16, 8, 16, decodes=4, ctx=(17, 128), lens=1, name="decode_tiny"),
        # A few short prompts at once (Qwen3-0.6B heads): the prefill counterpart, still bound by latency.
        _case("prefill", "core", 16, 8, 256, seqs=4, new=(17, 511), lens=2, name="prefill_tiny"),
        # One user's prompt on an idle server: its time to the first token (Qwen3-8B heads, 16-token pages).
        _case("prefill", "core", 32, 8, 16, seqs=1, new=(1999, 1999), lens=3, name="prefill_one_prompt"),
        # The next turns of two long conversations, each behind its own cached context (Qwen3-8B heads).
        _case("prefill", "core", 32, 8, 256, seqs=2, new=(128, 400), prefix=(6000, 15000), lens=4,
              name="prefill_turn"),
        # Prefix caching: a batch of new turns behind a common cached document (Qwen3-8B heads).
        _case("prefill", "attention", 32, 8, 256, seqs=64, new=(128, 1024), prefix=(0, 4096), shared=True, lens=5,
              name="prefill_prefix"),
        # The largest: long documents (Qwen3-32B heads, 8k to 32k tokens each).
        _case("prefill", "attention", 64, 8, 256, seqs=8, new=(8192, 32768), lens=6, name="prefill_long"),
        # Other model families' head sizes: 64 plain, and 256 with the logit soft cap (through the kernel entry).
        _case("prefill", "attention", 32, 8, 256, head_dim=64, seqs=16, new=(1000, 3000), lens=7,
              name="prefill_head64"),
        _case("prefill", "kernel", 32, 8, 256, head_dim=256, seqs=16, new=(1000, 3000), soft_cap=50.0, lens=8,
              name="prefill_head256_cap"),
        # One user's long conversation: a single 32k-token context (Qwen3-8B heads).
        _case("decode", "attention", 32, 8, 64, decodes=1, ctx=(32768, 32768), lens=9, name="decode_one_long"),
        # The serving batch: 256 sequences of 512 to 8192 tokens (Qwen3-8B heads).
        _case("decode", "core", 32, 8, 256, decodes=256, ctx=(512, 8192), lens=10, name="decode_batch"),
        # A smaller batch over float8 pages (Qwen3-32B heads): half the cache's memory.
        _case("decode", "kernel", 64, 8, 64, pages="fp8", decodes=48, ctx=(200, 4000), lens=11, name="decode_fp8"),
        # A scheduler step that mixes new prompts with running sequences (Qwen3-0.6B heads).
        _case("mixed", "core", 16, 8, 256, seqs=32, new=(64, 2048), decodes=96, ctx=(256, 4096), lens=12,
              name="mixed_step"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case: any step, the head counts of the listed ones (and a multi-query-like 64 / 2), head sizes,
    page sizes and page types in use, lengths over the logarithm of their range."""
    step = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "mixed"])
    heads, kv_heads = rng.choice([(16, 8), (32, 8), (64, 8), (32, 8), (64, 2)])
    page = rng.choice([16, 32, 64, 256])
    head_dim, pages, cap = 128, "bf16", 0.0
    entry = rng.choice(["core", "attention"])
    option = rng.random()
    if option < 0.25:
        head_dim, entry = rng.choice([64, 80, 96, 256]), "attention"
    elif option < 0.40 and step != "mixed":
        pages, entry = rng.choice(["fp8", "int8"]) if step == "decode" else "fp8", "kernel"
    if step != "mixed" and rng.random() < 0.12:
        cap, entry = 50.0, "kernel"
    lens = rng.randrange(1 << 20)
    c = _case(step, entry, heads, kv_heads, page, head_dim=head_dim, pages=pages, soft_cap=cap, lens=lens)
    if step != "prefill":
        n = _log_int(rng, 1, 256 if step == "decode" else 96)
        hi = _log_int(rng, 32, max(64, min(32768, 1_200_000 // n)))
        c.update(decodes=n, ctx_lo=max(1, hi // rng.choice([1, 2, 16])), ctx_hi=hi)
    if step != "decode":
        n = _log_int(rng, 1, 64 if step == "prefill" else 32)
        hi = _log_int(rng, 16, max(32, min(16384 if step == "prefill" else 2048, 131072 // n)))
        c.update(seqs=n, new_lo=max(1, hi // rng.choice([1, 2, 8])), new_hi=hi)
        if rng.random() < 0.4:
            p = _log_int(rng, 64, max(128, min(16384, 262144 // n)))
            c.update(prefix_lo=p // rng.choice([1, 4]), prefix_hi=p, shared=rng.random() < 0.5)
        while work(c)["flops"] > 20e12:  # far below the largest listed case
            c.update(new_lo=max(1, c["new_lo"] // 2), new_hi=max(1, c["new_hi"] // 2))
    return c


def _lengths(case):
    """(decode contexts, prefill new lengths, prefill cached lengths)."""
    rng = random.Random(case["lens"])
    ctx = [rng.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(case["decodes"])]
    new = [rng.randint(case["new_lo"], case["new_hi"]) for _ in range(case["seqs"])]
    pre = [rng.randint(case["prefix_lo"], case["prefix_hi"]) for _ in range(case["seqs"])]
    return ctx, new, pre


def work(case):
    ctx, new, pre = _lengths(case)
    h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    row = 2 * hkv * (2 * d if case["pages"] == "bf16" else d + 4)  # K and V of one token in the pool
    tokens = len(ctx) + sum(new)
    stored = 0 if case["pages"] == "int8" else tokens  # new tokens come as bf16 k / v and go to the pool
    cached = sum(ctx) - (len(ctx) if stored else 0) + (max(pre, default=0) if case["shared"] else sum(pre))
    pairs = sum(ctx) + sum(n * p + n * (n + 1) // 2 for n, p in zip(new, pre))
    table = sum(-(-n // case["page_size"]) for n in ctx + [n + p for n, p in zip(new, pre)])
    return {"bytes": cached * row + stored * (row + 4 * hkv * d) + 4 * tokens * h * d + 4 * table,
            "flops": 4 * d * h * pairs}


def tolerance(case):
    """Outputs are bf16 rows of f32 sums whose weights P (and, in prefill, the scaled q) are rounded to bf16: 2.1e-3
    to 4.0e-3 off the 64-bit result over the listed cases and drawn ones, so about four times that."""
    return {"rel": 1.4e-2, "max": 0.15}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _randn(shape, gen, dev):
    """Unit normal values in bf16, what normalised q / k rows and projected v rows look like."""
    t = torch.empty(shape, dtype=torch.bfloat16, device=dev)
    flat = t.view(-1)
    step = 1 << 28
    for s in range(0, flat.numel(), step):
        n = min(step, flat.numel() - s)
        flat[s:s + n] = torch.randn(n, generator=gen, device=dev, dtype=torch.float32)
    return t


def _layout(case, gen, dev):
    """Block tables (-1 padded), slots, positions and lengths, as the engine's scheduler lays them out: sequences'
    pages in a random order over the pool, decode sequences first."""
    ctx, new, pre = _lengths(case)
    bs = case["page_size"]
    total = ctx + [n + p for n, p in zip(new, pre)]
    first = [n - 1 for n in ctx] + pre            # position of a sequence's first new token
    count = [1] * len(ctx) + new                  # its new tokens
    common = [0] * len(ctx) + ([p // bs for p in pre] if case["shared"] else [0] * len(pre))
    doc = max(common, default=0)
    own = [-(-n // bs) - c for n, c in zip(total, common)]
    num_pages = doc + sum(own)
    num_pages += num_pages // 8 + 1               # a pool is never quite full
    perm = torch.randperm(num_pages, generator=gen, device=dev).to(torch.int32).cpu().numpy()
    table = np.full((len(total), max(c + o for c, o in zip(common, own))), -1, np.int32)
    at = doc
    slots, positions = [], []
    for i, (c, o) in enumerate(zip(common, own)):
        table[i, :c] = perm[:c]
        table[i, c:c + o] = perm[at:at + o]
        at += o
        pos = np.arange(first[i], first[i] + count[i])
        positions.append(pos)
        slots.append(table[i, pos // bs].astype(np.int64) * bs + pos % bs)
    i32 = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.int32), device=dev)  # noqa: E731
    cu = lambda n: i32(np.concatenate([[0], np.cumsum(n)]))  # noqa: E731
    return dict(num_pages=num_pages, block_tables=i32(table), slot_mapping=i32(np.concatenate(slots)),
                input_positions=i32(np.concatenate(positions)), cu_q=cu(count), cu_k=cu(total), lens=i32(total),
                count=count, total=total, first=first, max_new=max(count))


def _bucket(n):
    return 1 << max(0, n - 1).bit_length()


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    m = _layout(case, gen, dev)
    h, hkv, d, bs, nb = case["heads"], case["kv_heads"], case["head_dim"], case["page_size"], m["num_pages"]
    tokens = sum(m["count"])
    s = dict(case=case, layout=m)
    pool = (2, nb, bs, hkv, d)
    if case["pages"] == "bf16":
        s["kv_cache"] = _randn(pool, gen, dev)
    elif case["pages"] == "fp8":
        s["codes"] = torch.empty(pool, dtype=torch.float8_e4m3fn, device=dev)
        s["scales"] = torch.empty((2, hkv, nb, bs), dtype=torch.float32, device=dev)
        # cached tokens written the way the engine writes them, by the quantising store
        step = max(1, (1 << 27) // (bs * hkv * d))
        for p in range(0, nb, step):
            n = min(step, nb - p) * bs
            slot = torch.arange(p * bs, p * bs + n, dtype=torch.int32, device=dev)
            pa.update_kv_cache_fp8(s["codes"], s["scales"], slot, _randn((n, hkv, d), gen, dev),
                                   _randn((n, hkv, d), gen, dev))
    else:
        s["codes"] = (_randn(pool, gen, dev) * 32).clamp_(-127, 127).to(torch.int8)
        s["scales"] = 1 / 32 * torch.rand((2, hkv, nb, bs), generator=gen, device=dev, dtype=torch.float32) + 1 / 64
    s["q"] = _randn((tokens, h, d), gen, dev)
    s["k"] = _randn((tokens, hkv, d), gen, dev)
    s["v"] = _randn((tokens, hkv, d), gen, dev)
    if case["entry"] == "core":
        s["q_norm"] = (1 + 0.1 * torch.randn(d, generator=gen, device=dev)).to(torch.bfloat16)
        s["k_norm"] = (1 + 0.1 * torch.randn(d, generator=gen, device=dev)).to(torch.bfloat16)
    if case["step"] == "prefill":
        s["meta"] = pa.PrefillAttentionMetadata(m["input_positions"], m["slot_mapping"], m["block_tables"], m["cu_q"],
                                                m["cu_k"], None, None, _bucket(m["max_new"]))
    elif case["step"] == "decode":
        s["meta"] = pa.DecodeAttentionMetadata(m["input_positions"], m["slot_mapping"], m["block_tables"], m["lens"])
    else:
        s["meta"] = pa.MixedAttentionMetadata(m["input_positions"], m["slot_mapping"], m["block_tables"], m["cu_q"],
                                              m["lens"], case["decodes"], m["max_new"])
    return s


def run(s):
    case, meta = s["case"], s["meta"]
    if case["entry"] == "core":
        kv, out = pa.qwen3_attention_core(s["kv_cache"], s["q"], s["k"], s["v"], s["q_norm"], s["k_norm"], meta, eps=EPS,
                                          rope_theta=ROPE_THETA)
        return {"out": out, "pool": kv}
    if case["entry"] == "attention":
        kv, out = pa.attention(s["kv_cache"], s["q"], s["k"], s["v"], meta)
        return {"out": out, "pool": kv}
    res = {}
    if case["pages"] == "bf16":
        res["pool"] = pages = pa.update_kv_cache(s["kv_cache"], meta.slot_mapping, s["k"], s["v"])
        more = {}
    else:
        pages = s["codes"]
        if case["pages"] == "fp8":
            pa.update_kv_cache_fp8(pages, s["scales"], meta.slot_mapping, s["k"], s["v"])
            res.update(pool=pages.view(torch.uint8), scales=s["scales"])
        more = dict(k_scales_pages=s["scales"][0], v_scales_pages=s["scales"][1])
    if case["soft_cap"]:
        more["attn_logits_soft_cap"] = case["soft_cap"]
    k_pages, v_pages = pages[0].permute(2, 0, 1, 3), pages[1].permute(2, 0, 1, 3)
    if case["step"] == "decode":
        res["out"] = pa.decode_paged_attention(s["q"], k_pages, v_pages, meta.block_tables, meta.context_lens,
                                               scale=case["head_dim"] ** -0.5, **more)
    else:
        res["out"] = pa.prefill_paged_attention(s["q"], k_pages, v_pages, meta.block_tables, meta.cu_seqlens_q,
                                                meta.slot_mapping, meta.input_positions,
                                                max_seqlen_bucket=meta.max_seqlen_bucket,
                                                cu_seqlens_k=meta.cu_seqlens_k, **more)
    return res


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _bf16(x):
    return x.to(torch.bfloat16).to(torch.float64)


def _norm_rope(x, w, positions):
    """RMSNorm and RoPE over interleaved pairs; the rotation table is the model's, in bf16, the rest 64-bit."""
    d = x.shape[-1]
    x = x.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
    e = _bf16(torch.arange(0, d, 2, device=x.device, dtype=torch.float32) / d)
    inv = _bf16(1 / _bf16(_bf16(torch.tensor(ROPE_THETA, device=x.device, dtype=torch.float32)) ** e))
    f = _bf16(_bf16(positions.float())[:, None] * inv)
    cos, sin = _bf16(torch.cos(f))[:, None], _bf16(torch.sin(f))[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(x.shape)


def _attend(q, k, v, first, scale, cap):
    """q [n, H, d] at kv positions first .. first + n - 1, k / v [L, Hkv, d]: causal attention in 64 bits."""
    n, h, d = q.shape
    hkv = k.shape[1]
    g = h // hkv
    kt = k.permute(1, 2, 0).contiguous()                   # [Hkv, d, L]
    vt = v.permute(1, 0, 2).contiguous()                   # [Hkv, L, d]
    out = torch.empty_like(q)
    step = max(1, (1 << 29) // (h * k.shape[0]))
    for r in range(0, n, step):
        e = min(n, r + step)
        hi = min(k.shape[0], first + e)
        rows = q[r:e].reshape(e - r, hkv, g, d).permute(1, 2, 0, 3).reshape(hkv, g * (e - r), d)
        x = torch.matmul(rows, kt[:, :, :hi].contiguous()).mul_(scale)
        if cap:
            x = x.div_(cap).tanh_().mul_(cap)
        if e - r > 1:
            pos = torch.arange(first + r, first + e, device=q.device)
            hidden = torch.arange(hi, device=q.device)[None, :] > pos[:, None]
            x.view(hkv, g, e - r, hi).masked_fill_(hidden, float("-inf"))
        x.sub_(x.amax(-1, keepdim=True)).exp_()
        o = torch.matmul(x, vt[:, :hi].contiguous()) / x.sum(-1, keepdim=True)
        out[r:e] = o.view(hkv, g, e - r, d).permute(2, 0, 1, 3).reshape(e - r, h, d)
    return out


def exact(case, seed):
    s = prepare(case, seed)
    m, d, bs = s["layout"], case["head_dim"], case["page_size"]
    q, k, v = s["q"].double(), s["k"].double(), s["v"].double()
    if case["entry"] == "core":
        q = _norm_rope(s["q"], s["q_norm"], m["input_positions"])
        k = _norm_rope(s["k"], s["k_norm"], m["input_positions"])
    slots = m["slot_mapping"].long()
    res = {}
    if case["pages"] == "bf16":
        pool = s["kv_cache"].double().flatten(1, 2)        # [2, slots, Hkv, d]
        pool[0, slots], pool[1, slots] = k, v
        res["pool"] = pool.view(s["kv_cache"].shape)
        page = lambda ids: pool.unflatten(1, (-1, bs))[:, ids].flatten(1, 2)  # noqa: E731
    else:
        kind = s["codes"].dtype
        codes, scales = s["codes"].view(torch.uint8).flatten(1, 2), s["scales"].flatten(2, 3)
        if case["pages"] == "fp8":
            for i, x in enumerate((k, v)):
                top = x.abs().amax(-1).clamp_min(2.0 ** -118)
                e = torch.ceil(torch.log2(top / 448))
                codes[i, slots] = (x / torch.exp2(e)[..., None]).float().to(kind).view(torch.uint8)
                scales[i][:, slots] = torch.exp2(e).float().t()
            res.update(pool=None, scales=scales.view(s["scales"].shape).double())
        codes, scales = codes.unflatten(1, (-1, bs)), scales.unflatten(2, (-1, bs))

        def page(ids):
            w = scales[:, :, ids].double().permute(0, 2, 3, 1)[..., None]
            return (codes[:, ids].view(kind).float().double() * w).flatten(1, 2)

    # the scale as each entry applies it: prefill bf16(1 / sqrt d), decode 1 / bf16(sqrt d) (kernel entry: as given)
    root = torch.tensor(float(d) ** 0.5)
    pre_scale = float(_bf16(1 / root))
    dec_scale = d ** -0.5 if case["entry"] == "kernel" else 1 / float(_bf16(root))
    out = torch.empty_like(q)
    at = 0
    for i, (n, total, first) in enumerate(zip(m["count"], m["total"], m["first"])):
        ids = m["block_tables"][i, :-(-total // bs)].long()
        ctx = page(ids)[:, :total]
        scale = dec_scale if i < case["decodes"] else pre_scale
        out[at:at + n] = _attend(q[at:at + n], ctx[0], ctx[1], first, scale, case["soft_cap"])
        at += n
    res["out"] = out
    return res
