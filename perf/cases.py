"""The calls whose speed counts: paged attention as a serving loop makes them.

Five kinds of call, each through the package's public operators:

  decode  one new token per sequence over its paged context, alone or as a
          whole step (fill_kv_pages of the new tokens, then the attention)
  prompt  paged_attention_prefill: equal prompts over a paged history, the
          prompt's keys and values still in their projection rows
  chunk   chunked prefill: fill_kv_pages of ragged new chunks, then their
          causal attention through paged_attention
  mixed   one paged_attention call over decode rows and prefill chunks
  rope    rope_fill_kv_pages: rotate, cast and scatter a batch's new rows

Keys, values and queries are N(0, 1) unless a case asks for key outliers;
pages are randomly permuted in a pool with about 10 % free pages.  The
lengths of a ragged batch follow from the case alone (its ``lens_seed``), the
values and the page table from the seed given to ``prepare``.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path.cwd() / "proxy-attention-lab_amd"))

import proxy_attention_lab as pal  # noqa: E402

DEVICE = "cuda:0"
_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
_FP8 = torch.float8_e4m3fn

# 32 query heads on 8 kv heads of dimension 128 over 16-token pages is the
# shape of most of the benchmark's workloads
_BASE = {"hq": 32, "hkv": 8, "hd": 128, "tpp": 16, "dtype": "bf16", "fp8": False, "lens_seed": 1}


def _case(name: str, kind: str, **values) -> dict:
    return {"name": name, "kind": kind, **_BASE, **values}


def listed() -> list[dict]:
    return [
        # a handful of short requests on a small model: launches and latency
        _case("decode_tiny", "decode", seqs=4, ctx_lo=64, ctx_hi=256, hq=4, hkv=1, hd=64, dtype="f16",
              partition=0, fill=False, outliers=False),
        # one user in a chat of about three thousand tokens: latency of a token
        _case("decode_single", "decode", seqs=1, ctx_lo=3001, ctx_hi=3001, partition=0, fill=False, outliers=False),
        # the serving step of a full batch: write the new tokens, then attend
        _case("decode_step_64", "decode", seqs=64, ctx_lo=512, ctx_hi=4096, partition=0, fill=True, outliers=False),
        # the same batch over an fp8 cache
        _case("decode_fp8_64", "decode", seqs=64, ctx_lo=512, ctx_hi=4096, fp8=True, partition=0, fill=False,
              outliers=False),
        # a large batch of short contexts (classification, short answers)
        _case("decode_short_2048", "decode", seqs=2048, ctx_lo=16, ctx_hi=256, partition=0, fill=False,
              outliers=False),
        # long documents with a peaked softmax, in the two-pass form
        _case("decode_long_512", "decode", seqs=8, ctx_lo=32768, ctx_hi=131072, partition=512, fill=False,
              outliers=True),
        # a single prompt, nothing cached: time to the first token
        _case("prompt_single", "prompt", seqs=1, prompt=777, hist_lo=0, hist_hi=0),
        # equal prompts on cached histories
        _case("prompt_16", "prompt", seqs=16, prompt=1024, hist_lo=0, hist_hi=2048),
        # chunked prefill of a ragged batch
        _case("chunk_16", "chunk", seqs=16, new_lo=512, new_hi=2048, cached_lo=0, cached_hi=2048),
        # chunked prefill over an fp8 cache
        _case("chunk_fp8", "chunk", seqs=8, new_lo=256, new_hi=1024, cached_lo=0, cached_hi=4096, fp8=True),
        # decode rows and prefill chunks in one call (continuous batching)
        _case("mixed_f16", "mixed", seqs=256, ctx_lo=256, ctx_hi=8192, chunks=4, new=1024, cached_lo=0,
              cached_hi=4096, hq=64, dtype="f16"),
        # the projection's fp32 rows of a chunked prefill into the cache
        _case("rope_fill", "rope", seqs=16, new_lo=512, new_hi=2048, cached_lo=0, cached_hi=2048),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "decode", "prompt", "chunk", "mixed", "rope"])
    hq, hkv = rng.choice([(32, 8), (32, 8), (64, 8), (28, 4), (32, 32), (16, 2)])
    case = {"kind": kind, "hq": hq, "hkv": hkv, "hd": rng.choice([64, 128, 128, 128, 256]),
            "tpp": rng.choice([16, 16, 32]), "dtype": rng.choice(["bf16", "bf16", "f16"]),
            "fp8": rng.random() < 0.3, "lens_seed": rng.randrange(1, 1 << 30)}
    token_bytes = 4 * hkv * case["hd"]  # K and V of a token, 16 bit
    if kind == "decode":
        seqs = _log_int(rng, 1, 2048)
        # the batch's context up to 2 GB of 16-bit K and V
        hi = min(131072, int(2e9 / (token_bytes * seqs)))
        ctx_hi = _log_int(rng, min(48, hi), hi)
        case.update(seqs=seqs, ctx_lo=max(1, ctx_hi // rng.choice([1, 2, 8])), ctx_hi=ctx_hi,
                    partition=rng.choice([0, 0, 0, 512]), fill=rng.random() < 0.5, outliers=rng.random() < 0.2)
    elif kind == "mixed":
        case.update(seqs=_log_int(rng, 4, 256), ctx_lo=rng.randrange(1, 512), ctx_hi=_log_int(rng, 512, 4096),
                    chunks=rng.randrange(1, 5), new=_log_int(rng, 16, 1024), cached_lo=0,
                    cached_hi=rng.randrange(0, 4097))
        while case["seqs"] * case["ctx_hi"] * token_bytes > 3e9:
            case["ctx_hi"] = max(513, case["ctx_hi"] // 2)
            case["seqs"] = max(4, case["seqs"] // 2)
    else:
        seqs = _log_int(rng, 1, 16)
        new_hi = _log_int(rng, 16, 2048)
        cached_hi = rng.randrange(0, 2049)
        if kind == "prompt":
            case.update(seqs=seqs, prompt=new_hi, hist_lo=0, hist_hi=cached_hi)
        else:
            case.update(seqs=seqs, new_lo=max(1, new_hi // 4), new_hi=new_hi, cached_lo=0, cached_hi=cached_hi)
        # no more attention work than the largest listed chunk
        while work(case)["flops"] > 5e11 or case["seqs"] * new_hi * hq * case["hd"] > 1.2e8:
            new_hi = max(16, new_hi // 2)
            case.update({"prompt": new_hi} if kind == "prompt" else {"new_lo": max(1, new_hi // 4), "new_hi": new_hi})
    return case


# ---------------------------------------------------------------------------
# shapes of a case
# ---------------------------------------------------------------------------


def _between(rng, lo: int, hi: int, n: int) -> np.ndarray:
    return rng.integers(lo, hi + 1, size=n).astype(np.int32)


def _lengths(case: dict) -> tuple[np.ndarray, np.ndarray]:
    """(tokens already cached, new tokens) of each sequence."""
    rng = np.random.default_rng(case["lens_seed"])
    n = case["seqs"]
    if case["kind"] == "decode":
        return _between(rng, case["ctx_lo"], case["ctx_hi"], n) - 1, np.ones(n, np.int32)
    if case["kind"] == "prompt":
        return _between(rng, case["hist_lo"], case["hist_hi"], n), np.full(n, case["prompt"], np.int32)
    if case["kind"] == "mixed":
        dec = _between(rng, case["ctx_lo"], case["ctx_hi"], n) - 1
        cached = _between(rng, case["cached_lo"], case["cached_hi"], case["chunks"])
        return (np.concatenate([dec, cached]),
                np.concatenate([np.ones(n, np.int32), np.full(case["chunks"], case["new"], np.int32)]))
    return (_between(rng, case["cached_lo"], case["cached_hi"], n),
            _between(rng, case["new_lo"], case["new_hi"], n))


def work(case: dict) -> dict:
    cached, new = (x.astype(np.float64) for x in _lengths(case))
    hq, hkv, hd, tpp = case["hq"], case["hkv"], case["hd"], case["tpp"]
    el = 1 if case["fp8"] else 2
    rows = float(new.sum())
    kv_row = 2 * hkv * hd  # elements of a token's K and V
    if case["kind"] == "rope":  # fp32 rows in, 16-bit queries and pool rows out, a cos/sin row per token
        return {"bytes": rows * (kv_row * (4 + el) + hq * hd * (4 + 2) + hd * 4), "flops": rows * 6 * (hq + hkv) * hd}
    pairs = float((new * cached + new * (new + 1) / 2).sum())
    pool_tokens = cached if case["kind"] == "prompt" else cached + new
    total = float(pool_tokens.sum()) * kv_row * el + 2 * rows * hq * hd * 2
    if case["fp8"]:
        total += float(np.ceil(pool_tokens / tpp).sum()) * hkv * 2 * 4
    if case["kind"] == "prompt":
        total += rows * kv_row * 2
    elif case["kind"] == "chunk" or case.get("fill"):
        total += rows * kv_row * (2 + el)
    return {"bytes": total, "flops": 4.0 * hq * hd * pairs}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _randn(g: torch.Generator, shape, dtype: torch.dtype) -> torch.Tensor:
    return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32).to(dtype)


def _pools(case: dict, g: torch.Generator, pages: int) -> dict:
    dtype = _DTYPES[case["dtype"]]
    hkv, hd, tpp = case["hkv"], case["hd"], case["tpp"]
    if not case["fp8"]:
        return {"k_pool": _randn(g, pal.get_k_cache_shape(pages, hkv, hd, tpp, dtype), dtype),
                "v_pool": _randn(g, pal.get_v_cache_shape(pages, hkv, hd, tpp, dtype), dtype), "scales": {}}
    out = {"scales": {}}
    for key, shape in (("k", pal.get_k_cache_shape(pages, hkv, hd, tpp, _FP8)),
                       ("v", pal.get_v_cache_shape(pages, hkv, hd, tpp, _FP8))):
        # the scale a calibration over N(0, 1) rows gives: about 1.2 to 2 x (largest value) / 448
        scale = torch.rand((pages, hkv), generator=g, device=DEVICE) * 0.008 + 0.012
        x = torch.randn(shape, generator=g, device=DEVICE)
        out[f"{key}_pool"] = (x / scale.view((pages, hkv) + (1,) * (x.dim() - 2))).clamp(-448, 448).to(_FP8)
        out["scales"][f"{key}_scales"] = scale
    return out


def prepare(case: dict, seed: int) -> dict:
    rng = np.random.default_rng([case["lens_seed"], seed])
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(rng.integers(1 << 62)))
    dtype = _DTYPES[case["dtype"]]
    hq, hkv, hd, tpp, kind = case["hq"], case["hkv"], case["hd"], case["tpp"], case["kind"]
    cached, new = _lengths(case)
    held = cached if kind == "prompt" else cached + new  # tokens with a slot in the pool
    per_seq = (held.astype(np.int64) + tpp - 1) // tpp
    used = int(per_seq.sum())
    pages = max(1, used + math.ceil(0.1 * used))
    table = np.zeros((len(held), max(1, int(per_seq.max()))), np.int32)
    perm = rng.permutation(pages).astype(np.int32)
    ends = np.cumsum(per_seq)
    for s, (n, end) in enumerate(zip(per_seq, ends)):
        table[s, :n] = perm[end - n:end]
    st = _pools(case, g, pages)
    st.update(case=case, page_table=torch.from_numpy(table).to(DEVICE), cached=cached, new=new)

    if case.get("outliers") and not case["fp8"]:  # 1 % of the key rows x 8
        hot = [rng.choice(int(n), size=max(1, int(n) // 100), replace=False) for n in held]
        page = torch.from_numpy(np.concatenate([table[s, p // tpp] for s, p in enumerate(hot)]).astype(np.int64))
        slot = torch.from_numpy(np.concatenate([p % tpp for p in hot]).astype(np.int64))
        page, slot = page.to(DEVICE), slot.to(DEVICE)
        st["k_pool"][page, :, :, slot, :] = st["k_pool"][page, :, :, slot, :] * 8

    if kind == "mixed":
        # every decode row is a block of its own, chunks come in blocks of up
        # to 128 rows, and the blocks arrive in random order
        blocks = [(s, int(cached[s]), 1) for s in range(case["seqs"])]
        for s in range(case["seqs"], len(new)):
            blocks += [(s, int(cached[s]) + b, min(128, int(new[s]) - b)) for b in range(0, int(new[s]), 128)]
        blocks = [blocks[i] for i in rng.permutation(len(blocks))]
        q2s = np.concatenate([np.full(n, s, np.int32) for s, _, n in blocks])
        pos = np.concatenate([np.arange(p, p + n, dtype=np.int32) for _, p, n in blocks])
    else:
        q2s = np.repeat(np.arange(len(new), dtype=np.int32), new)
        pos = np.concatenate([np.arange(c, c + n, dtype=np.int32) for c, n in zip(cached, new)])
    rows = len(q2s)
    st["rows"], st["q2s_host"], st["pos_host"] = rows, q2s, pos
    st["seq_lens"] = torch.from_numpy(held.astype(np.int32)).to(DEVICE)
    st["q2s"] = torch.from_numpy(q2s).to(DEVICE)
    st["pos"] = torch.from_numpy(pos).to(DEVICE)
    st["offset"] = torch.from_numpy(pos + 1).to(DEVICE)
    row_dtype = torch.float32 if kind == "rope" else dtype
    st["queries"] = _randn(g, (rows, hq, hd), row_dtype)
    if kind in ("prompt", "chunk", "rope") or case.get("fill"):
        st["new_k"] = _randn(g, (rows, hkv, hd), row_dtype)
        st["new_v"] = _randn(g, (rows, hkv, hd), row_dtype)
    if kind == "rope":
        half = hd // 2
        ang = torch.arange(int(held.max()), dtype=torch.float64, device=DEVICE)[:, None] * \
            500000.0 ** (-2.0 * torch.arange(half, dtype=torch.float64, device=DEVICE) / hd)[None, :]
        st["cos_sin"] = torch.cat([torch.cos(ang), torch.sin(ang)], dim=1).to(torch.float32)
    # what a pass hands back of the pools it wrote (fp8 codes as bytes)
    st["k_out"], st["v_out"] = (t.view(torch.uint8) if case["fp8"] else t for t in (st["k_pool"], st["v_pool"]))
    return st


def _fill(st: dict) -> None:
    pal.fill_kv_pages(st["new_k"], st["new_v"], st["k_pool"], st["v_pool"], st["page_table"], st["pos"], st["q2s"],
                      **st["scales"])


def run(st: dict):
    case = st["case"]
    kind = case["kind"]
    if kind == "prompt":
        return pal.paged_attention_prefill(st["queries"], st["new_k"], st["new_v"], st["k_pool"], st["v_pool"],
                                           st["page_table"], st["seq_lens"], **st["scales"])
    if kind == "rope":
        _, _, q = pal.rope_fill_kv_pages(st["new_k"], st["new_v"], st["k_pool"], st["v_pool"], st["page_table"],
                                         st["pos"], st["q2s"], st["cos_sin"], queries=st["queries"],
                                         query_dtype=_DTYPES[case["dtype"]], **st["scales"])
        return q, st["k_out"], st["v_out"]
    if kind == "decode":
        if case["fill"]:
            _fill(st)
        out = pal.paged_attention_decode(st["queries"], st["k_pool"], st["v_pool"], st["page_table"],
                                         st["seq_lens"], partition_size=case["partition"], **st["scales"])
        return (out, st["k_out"], st["v_out"]) if case["fill"] else out
    if kind == "chunk":
        _fill(st)
    out = pal.paged_attention(st["queries"], st["k_pool"], st["v_pool"], st["page_table"], st["seq_lens"], st["q2s"],
                              st["offset"], **st["scales"])
    return (out, st["k_out"], st["v_out"]) if kind == "chunk" else out


def tolerance(case: dict):
    if case["kind"] == "rope":
        return "exact"  # one rounding of each product as written: the pools are held bit for bit
    # Against float64 the path shows 1.7e-3 to 3.2e-3 in bf16 and 2.6e-4 to
    # 3.6e-4 in fp16 (output, probabilities and partials rounded to 16 bits),
    # its single values up to 0.031 and 0.0027 of the output's root mean square.
    if case["dtype"] == "f16":
        return {"rel": 1.5e-3, "max": 1.1e-2}
    return {"rel": 1e-2, "max": 1.2e-1}


# ---------------------------------------------------------------------------
# the same in 64 bits, without the package
# ---------------------------------------------------------------------------


def _write_rows(st: dict, k_new: torch.Tensor, v_new: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """Copies of the pools as [pages, tpp, hkv, hd] values in the pool's
    precision (fp8: its codes' values) with the new rows written."""
    case = st["case"]
    k, v = st["k_pool"], st["v_pool"]
    pages, hkv, hd, tpp = v.shape
    if case["fp8"]:
        k, v = k.to(torch.float32), v.to(torch.float32)
    k = k.permute(0, 3, 1, 2, 4).reshape(pages, tpp, hkv, hd).clone()
    v = v.permute(0, 3, 1, 2).contiguous()
    if k_new is not None:
        page = st["page_table"][st["q2s"].long(), (st["pos"] // tpp).long()].long()
        slot = (st["pos"] % tpp).long()
        for pool, new, sc in ((k, k_new, "k_scales"), (v, v_new, "v_scales")):
            if case["fp8"]:
                new = (new.float() / st["scales"][sc][page][:, :, None]).clamp(-448, 448).to(_FP8).to(torch.float32)
            pool[page, slot] = new.to(pool.dtype)
    return k, v


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, limits: torch.Tensor) -> torch.Tensor:
    """Rows q [n, hq, hd] over keys k, v [t, hkv, hd]; row i sees limits[i] keys."""
    n, hq, hd = q.shape
    hkv = k.shape[1]
    grp = hq // hkv
    out = torch.empty((n, hq, hd), dtype=torch.float64, device=q.device)
    hidden = None if n == 1 else torch.arange(k.shape[0], device=q.device)[None, :] >= limits[:, None]
    for h in range(hkv):
        qh = q[:, h * grp:(h + 1) * grp].double().transpose(0, 1).reshape(grp * n, hd)
        s = torch.matmul(qh, k[:, h].double().t().contiguous()) / math.sqrt(hd)
        if hidden is not None:
            s = s.view(grp, n, -1).masked_fill_(hidden[None], -math.inf).view(grp * n, -1)
        o = torch.matmul(torch.softmax(s, dim=1), v[:, h].double().contiguous())
        out[:, h * grp:(h + 1) * grp] = o.view(grp, n, hd).transpose(0, 1)
    return out


def _rotated(st: dict, x: torch.Tensor) -> torch.Tensor:
    half = x.shape[-1] // 2
    cs = st["cos_sin"][st["pos"].long()].double()[:, None, :]
    cos, sin = cs[..., :half], cs[..., half:]
    a, b = x[..., :half].double(), x[..., half:].double()
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _pool_layout(case: dict, k: torch.Tensor, v: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    pages, tpp, hkv, hd = k.shape
    k = k.double().view(pages, tpp, hkv, hd // 8, 8).permute(0, 2, 3, 1, 4).contiguous()
    return k, v.double().permute(0, 2, 3, 1).contiguous()


def exact(case: dict, seed: int):
    st = prepare(case, seed)
    kind, tpp = case["kind"], case["tpp"]
    if kind == "rope":
        q = _rotated(st, st["queries"])
        if case["fp8"]:
            return q, None, None
        k, v = _write_rows(st, None, None)
        k, v = k.double(), v.double()
        page = st["page_table"][st["q2s"].long(), (st["pos"] // tpp).long()].long()
        slot = (st["pos"] % tpp).long()
        k[page, slot] = _rotated(st, st["new_k"])
        v[page, slot] = st["new_v"].double()
        return (q, *_pool_layout(case, k, v))
    filled = kind == "chunk" or bool(case.get("fill"))
    k_all, v_all = _write_rows(st, st["new_k"] if filled else None, st["new_v"] if filled else None)
    out = torch.empty((st["rows"], case["hq"], case["hd"]), dtype=torch.float64, device=DEVICE)
    order = np.argsort(st["q2s_host"], kind="stable")
    bounds = np.searchsorted(st["q2s_host"][order], np.arange(len(st["new"]) + 1))
    held = st["seq_lens"].cpu().numpy()
    for s in range(len(st["new"])):
        n = int(held[s])
        pages = st["page_table"][s, :(n + tpp - 1) // tpp].long()
        k, v = k_all[pages], v_all[pages]
        if case["fp8"]:
            k = k.double() * st["scales"]["k_scales"][pages].double()[:, None, :, None]
            v = v.double() * st["scales"]["v_scales"][pages].double()[:, None, :, None]
        k, v = k.flatten(0, 1)[:n], v.flatten(0, 1)[:n]
        if kind == "prompt":
            p0 = s * case["prompt"]
            k = torch.cat([k.double(), st["new_k"][p0:p0 + case["prompt"]].double()])
            v = torch.cat([v.double(), st["new_v"][p0:p0 + case["prompt"]].double()])
        rows = torch.from_numpy(order[bounds[s]:bounds[s + 1]]).to(DEVICE)
        out[rows] = _attend(st["queries"][rows], k, v, st["offset"][rows])
    if kind == "prompt":
        return out.view(-1, case["hd"])
    if not filled:
        return out
    if case["fp8"]:
        return out, None, None
    return (out, *_pool_layout(case, k_all, v_all))
