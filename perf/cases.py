"""Timed cases of the paged-KV attention path: what they are, their inputs, one pass of each, and its exact result.

Every pass goes through the public Python entry points (`oxide_paged_kv`), which call the C ABI.  Shapes are the
repository's benchmark configurations and the head layouts that its header and tests name; caches hold N(0, 1)
values in pages handed out in a random order.  Sequence lengths belong to the case (so that its work is known
without a seed); values, queries and the order of the pages come from the seed.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PACKAGE_PARENT = str(Path.cwd() / "vllm-oxide_amd")
if _PACKAGE_PARENT not in sys.path:
    sys.path.insert(0, _PACKAGE_PARENT)

import oxide_paged_kv as ox  # noqa: E402

_DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16}
_EPS = 1e-6
_MAX_POSITION = 40960
_DEVICE = "cuda:0"

# Query heads, kv heads of Qwen3-0.6B, Qwen3-8B, Qwen3-14B, Qwen3-32B and Qwen2.5-7B.
_HEADS = ((16, 8), (32, 8), (40, 8), (64, 8), (28, 4))


def _decode(name, heads, kv_heads, batch, lo, hi, dim=128, dtype="bf16", page=256, window=-1, shared=0):
    return {"name": name, "kind": "decode", "heads": heads, "kv_heads": kv_heads, "dim": dim, "dtype": dtype,
            "batch": batch, "lo": lo, "hi": hi, "page": page, "window": window, "shared": shared}


def _prefill(name, heads, kv_heads, batch, lo, hi, cached_lo=0, cached_hi=0, paged=True, dim=128, dtype="bf16",
             page=256, window=-1):
    return {"name": name, "kind": "prefill", "heads": heads, "kv_heads": kv_heads, "dim": dim, "dtype": dtype,
            "batch": batch, "lo": lo, "hi": hi, "cached_lo": cached_lo, "cached_hi": cached_hi, "paged": paged,
            "page": page, "window": window}


def listed():
    return [
        # The smallest decode step: one layer of a small model for four users, all three calls an engine makes --
        # metadata on the device, the fused q/k norm + rotation + append, then attention.
        {"name": "layer_step_b4", "kind": "layer", "heads": 16, "kv_heads": 8, "dim": 128, "dtype": "bf16",
         "batch": 4, "lo": 300, "hi": 1000, "page": 256},
        # One user with a long conversation: a single sequence has to fill the whole chip.
        _decode("decode_single_32k", 32, 8, 1, 32000, 32768),
        # The 0.6B benchmark batch: many short ragged sequences.
        _decode("decode_0.6b_b32", 16, 8, 32, 512, 4096),
        # The headline: the 8B serving batch.
        _decode("decode_8b_b64", 32, 8, 64, 2048, 8192),
        # Long documents on the 32B head layout; the largest pass.
        _decode("decode_32b_b16_long", 64, 8, 16, 32768, 131072),
        # Many users of one system prompt: 15 whole shared pages, then own tokens, sliding window.
        _decode("decode_shared_prefix_b128", 32, 8, 128, 4096 + 64, 4096 + 1024, window=4096, shared=3840),
        # Ragged mid-size batch in f16 with small pages, a sliding window and an odd group (five).
        _decode("decode_14b_f16_window", 40, 8, 23, 100, 6000, dtype="f16", page=16, window=2047),
        # Prompts prefilled in full over the paged cache.
        _prefill("prefill_8b_4x4096", 32, 8, 4, 4096, 4096),
        # A batch of short ragged prompts over contiguous K/V.
        _prefill("prefill_ragged_short", 16, 8, 16, 64, 1500, paged=False),
        # Chunked prefill / prefix hits: a few hundred new tokens each behind long cached contexts.
        _prefill("prefill_chunk_cached", 32, 8, 2, 250, 512, cached_lo=8000, cached_hi=24000),
        # The attention prologue of a prefill step (8B heads).
        {"name": "prologue_16k", "kind": "prologue", "heads": 32, "kv_heads": 8, "dim": 128, "dtype": "bf16",
         "tokens": 16384, "page": 256},
        # Copy-on-write of shared pages and the gather of a prefix hit.
        {"name": "block_moves", "kind": "blocks", "kv_heads": 8, "dim": 128, "dtype": "bf16", "page": 256,
         "pairs": 128, "gathered": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("layer", "decode", "decode", "decode", "prefill", "prefill", "prefill", "prologue", "blocks"))
    heads, kv_heads = rng.choice(_HEADS)
    dim = rng.choice((128, 128, 128, 64))
    dtype = rng.choice(("bf16", "bf16", "f16"))
    page = rng.choice((256, 256, 64, 16))
    case = {"kind": kind, "heads": heads, "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "page": page}
    if kind in ("layer", "decode"):
        batch = _log_int(rng, 1, 128)
        # At most the long 32B case's keys in total, and positions inside the rotation table for a layer.
        hi = _log_int(rng, 64, min(131072 if kind == "decode" else _MAX_POSITION - 1, 1_000_000 // batch))
        lo = max(1, int(hi * rng.choice((0.1, 0.25, 0.9))))
        case.update(batch=batch, lo=lo, hi=hi)
        if kind == "decode":
            window = rng.choice((-1, -1, -1, max(1, hi // 2)))
            shared = lo // page // 2 * page if batch > 1 and rng.random() < 0.25 else 0
            case.update(window=window, shared=shared)
    elif kind == "prefill":
        batch = _log_int(rng, 1, 16)
        hi = _log_int(rng, 16, 4096)
        lo = max(1, int(hi * rng.choice((0.1, 0.5, 1.0))))
        cached_hi = rng.choice((0, _log_int(rng, 256, 24000)))
        # At most the listed 4 x 4096 case's query-key-head products.
        while batch * heads * hi * (cached_hi + hi / 2) > 4 * 32 * 4096 * 2048:
            cached_hi //= 2
            hi = max(16, hi * 3 // 4)
            lo = min(lo, hi)
        paged = cached_hi > 0 or rng.random() < 0.5
        case.update(batch=batch, lo=lo, hi=hi, cached_lo=cached_hi // 3, cached_hi=cached_hi, paged=paged,
                    window=rng.choice((-1, -1, -1, max(1, hi // 2))))
    elif kind == "prologue":
        case.update(tokens=_log_int(rng, 1, 16384))
    else:
        del case["heads"]
        case.update(pairs=_log_int(rng, 1, 256), gathered=_log_int(rng, 1, 256))
    return case


def _lengths(lo, hi, n, salt):
    """n lengths in [lo, hi] with both ends among them, the same for every seed."""
    r = np.random.default_rng([salt, lo, hi, n])
    out = r.integers(lo, hi, size=n, endpoint=True)
    out[r.integers(0, n)] = hi
    return out


def _generator(seed):
    g = torch.Generator(device=_DEVICE)
    g.manual_seed(int(seed))
    return g


def _normal(shape, dtype, g):
    return torch.randn(shape, dtype=dtype, device=_DEVICE, generator=g)


def _pages(lengths, page, seed, shared_pages=0):
    """Block table [n, width] (rows padded with 0), the pool's size, and the ragged rows: pages in a random order,
    the first shared_pages the same in every row."""
    counts = [(int(x) + page - 1) // page for x in lengths]
    need = shared_pages + sum(c - shared_pages for c in counts)
    pool = need + 16
    order = np.random.default_rng(int(seed)).permutation(pool).astype(np.int32)
    table = np.zeros((len(counts), max(max(counts), 1)), np.int32)
    at = shared_pages
    for i, c in enumerate(counts):
        table[i, :shared_pages] = order[:shared_pages]
        table[i, shared_pages:c] = order[at:at + c - shared_pages]
        at += c - shared_pages
    return table, pool


def _prefix_sums(lengths):
    out = np.zeros(len(lengths) + 1, np.int32)
    out[1:] = np.cumsum(lengths)
    return torch.from_numpy(out).to(_DEVICE)


def _slots(table, lengths, page):
    """Slot of each sequence's newest token."""
    return np.array([int(table[i, (x - 1) // page]) * page + int((x - 1) % page) for i, x in enumerate(lengths)],
                    np.int64)


def _rope_table(dim):
    """fp32 [position, cos | sin] at base 1e6."""
    f = 1e6 ** (-torch.arange(0, dim, 2, dtype=torch.float64, device=_DEVICE) / dim)
    a = torch.arange(_MAX_POSITION, dtype=torch.float64, device=_DEVICE)[:, None] * f
    return torch.cat([a.cos(), a.sin()], 1).float()


def _caches(case, pool, g):
    shape = (pool, case["page"], case["kv_heads"], case["dim"])
    dt = _DTYPE[case["dtype"]]
    return _normal(shape, dt, g), _normal(shape, dt, g)


def prepare(case, seed):
    g = _generator(seed)
    kind, dim = case["kind"], case["dim"]
    dt = _DTYPE[case["dtype"]]
    s = {"case": case, "scale": 1.0 / math.sqrt(dim)}
    if kind in ("layer", "decode"):
        heads, kv_heads, n = case["heads"], case["kv_heads"], case["batch"]
        lengths = _lengths(case["lo"], case["hi"], n, 1)
        table, pool = _pages(lengths, case["page"], seed, case.get("shared", 0) // case["page"])
        s["table"] = torch.from_numpy(table).to(_DEVICE)
        s["longest"] = int(lengths.max())
        s["k_cache"], s["v_cache"] = _caches(case, pool, g)
        if kind == "layer":
            s["context_lens"] = torch.from_numpy(lengths.astype(np.int32)).to(_DEVICE)
            s["positions"] = torch.from_numpy(lengths.astype(np.int32) - 1).to(_DEVICE)
            s["qkv"] = _normal((n, (heads + 2 * kv_heads) * dim), dt, g)
            s["q_weight"], s["k_weight"] = (1 + 0.1 * _normal((dim,), torch.float32, g)).to(dt), \
                (1 + 0.1 * _normal((dim,), torch.float32, g)).to(dt)
            s["rope"] = _rope_table(dim)
        else:
            s["cu"] = _prefix_sums(lengths)
            s["q"] = _normal((n, heads, dim), dt, g)
            s["key"], s["value"] = _normal((n, kv_heads, dim), dt, g), _normal((n, kv_heads, dim), dt, g)
            s["slots"] = torch.from_numpy(_slots(table, lengths, case["page"])).to(_DEVICE)
    elif kind == "prefill":
        new, cached = _lengths(case["lo"], case["hi"], case["batch"], 2), \
            _lengths(case["cached_lo"], case["cached_hi"], case["batch"], 3)
        total = new + cached
        s["cu_q"], s["cu_k"] = _prefix_sums(new), _prefix_sums(total)
        s["longest_q"], s["longest_k"] = int(new.max()), int(total.max())
        s["q"] = _normal((int(new.sum()), case["heads"], dim), dt, g)
        if case["paged"]:
            table, pool = _pages(total, case["page"], seed)
            s["table"] = torch.from_numpy(table).to(_DEVICE)
            s["k_cache"], s["v_cache"] = _caches(case, pool, g)
        else:
            shape = (int(total.sum()), case["kv_heads"], dim)
            s["k"], s["v"] = _normal(shape, dt, g), _normal(shape, dt, g)
    elif kind == "prologue":
        heads, kv_heads, n = case["heads"], case["kv_heads"], case["tokens"]
        pool = (n + case["page"] - 1) // case["page"] + 2
        order = np.random.default_rng(int(seed)).permutation(pool)
        t = np.arange(n)
        s["slots"] = torch.from_numpy((order[t // case["page"]] * case["page"] + t % case["page"]).astype(np.int64)) \
            .to(_DEVICE)
        s["positions"] = torch.from_numpy(t.astype(np.int32)).to(_DEVICE)
        s["qkv"] = _normal((n, (heads + 2 * kv_heads) * dim), dt, g)
        s["q_weight"], s["k_weight"] = (1 + 0.1 * _normal((dim,), torch.float32, g)).to(dt), \
            (1 + 0.1 * _normal((dim,), torch.float32, g)).to(dt)
        s["rope"] = _rope_table(dim)
        s["k_cache"], s["v_cache"] = _caches(case, pool, g)
    else:
        pairs, gathered = case["pairs"], case["gathered"]
        pool = 2 * pairs + gathered + 16
        order = np.random.default_rng(int(seed)).permutation(pool).astype(np.int64)
        s["pairs"] = torch.from_numpy(np.ascontiguousarray(order[:2 * pairs].reshape(pairs, 2))).to(_DEVICE)
        s["ids"] = torch.from_numpy(order[2 * pairs:2 * pairs + gathered].astype(np.int32)).to(_DEVICE)
        s["k_cache"], s["v_cache"] = _caches(case, pool, g)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    window = None if case.get("window", -1) < 0 else case["window"]
    if kind == "decode":
        out = ox.decode_attn(s["q"], s["k_cache"], s["v_cache"], s["cu"], s["table"], s["longest"], s["scale"],
                             window_left=window, page_block_size=case["page"],
                             append=(s["key"], s["value"], s["slots"]),
                             shared_prefix_blocks=case["shared"] // case["page"] if case["shared"] else None)
        return out, s["k_cache"], s["v_cache"]
    if kind == "layer":
        cu, slots = ox.build_decode_metadata(s["context_lens"], s["table"], case["page"])
        q = ox.qk_norm_rope_and_cache(s["qkv"], case["heads"], case["kv_heads"], s["q_weight"], s["k_weight"], _EPS,
                                      s["rope"], s["positions"], s["k_cache"], s["v_cache"], slots)
        out = ox.decode_attn(q, s["k_cache"], s["v_cache"], cu, s["table"], s["longest"], s["scale"],
                             page_block_size=case["page"])
        return out, q, s["k_cache"], s["v_cache"], cu, slots
    if kind == "prefill":
        if case["paged"]:
            return ox.prefill_attn(s["q"], s["k_cache"], s["v_cache"], s["cu_q"], s["cu_k"], s["longest_q"],
                                   s["longest_k"], s["scale"], block_table=s["table"], window_left=window)
        return ox.prefill_attn(s["q"], s["k"], s["v"], s["cu_q"], s["cu_k"], s["longest_q"], s["longest_k"],
                               s["scale"], window_left=window)
    if kind == "prologue":
        q = ox.qk_norm_rope_and_cache(s["qkv"], case["heads"], case["kv_heads"], s["q_weight"], s["k_weight"], _EPS,
                                      s["rope"], s["positions"], s["k_cache"], s["v_cache"], s["slots"])
        return q, s["k_cache"], s["v_cache"]
    ox.copy_blocks(s["k_cache"], s["v_cache"], s["pairs"])
    k, v = ox.gather_blocks(s["k_cache"], s["v_cache"], s["ids"])
    return s["k_cache"], s["v_cache"], k, v


def work(case):
    kind, dim = case["kind"], case["dim"]
    kv_row = 2 * case["kv_heads"] * dim * 2  # bytes of one token's K and V rows
    if kind in ("decode", "layer"):
        lengths = _lengths(case["lo"], case["hi"], case["batch"], 1)
        window = case.get("window", -1)
        first = np.maximum(lengths - 1 - window, 0) if window >= 0 else np.zeros_like(lengths)
        shared = case.get("shared", 0)
        own = np.maximum(lengths - np.maximum(first, shared), 0).sum()
        common = max(0, shared - int(first.min())) if shared else 0  # read once for all
        n, q_row = case["batch"], case["heads"] * dim * 2
        moved = (int(own) + common) * kv_row + n * 2 * q_row + 2 * n * kv_row
        if kind == "layer":
            moved += n * (q_row + 3 * 8 + 8 * dim)  # merged row in, q written (and read back as an input), table rows
        return {"bytes": int(moved), "flops": int(4 * dim * case["heads"] * (lengths - first).sum())}
    if kind == "prefill":
        new, cached = _lengths(case["lo"], case["hi"], case["batch"], 2), \
            _lengths(case["cached_lo"], case["cached_hi"], case["batch"], 3)
        window, seen, keys = case["window"], 0, 0
        for a, c in zip(new.tolist(), cached.tolist()):
            visible = np.arange(c + 1, c + a + 1)
            if window >= 0:
                visible = np.minimum(visible, window + 1)
                keys += min(a + c, a + window)
            else:
                keys += a + c
            seen += int(visible.sum())
        return {"bytes": int(2 * new.sum() * case["heads"] * dim * 2 + keys * kv_row),
                "flops": int(4 * dim * case["heads"] * seen)}
    if kind == "prologue":
        n = case["tokens"]
        return {"bytes": int(n * (2 * case["heads"] * dim * 2 + 2 * kv_row + 4 * dim + 12)), "flops": 0}
    return {"bytes": int((case["pairs"] + case["gathered"]) * 2 * case["page"] * kv_row), "flops": 0}


def tolerance(case):
    # Measured against `exact`; the stated bounds are about four times what the start shows.  Attention rounds its
    # probabilities and its result to 16 bits (bf16 2^-9, f16 2^-12 at most each); a layer and the prologue also
    # round between the norm, the weight and the rotation.
    if case["kind"] == "blocks":
        return "exact"
    bf16 = case["dtype"] == "bf16"
    if case["kind"] == "layer":
        return {"rel": 1.6e-2 if bf16 else 2e-3}
    return {"rel": 1e-2 if bf16 else 1.3e-3}


def _attend(q, k, v, first, last, scale):
    """q [Lq, heads, D] over k / v [Lk, kv_heads, D] in float64; row i sees keys first[i] .. last[i]."""
    lq, heads, dim = q.shape
    kv_heads = k.shape[1]
    group = heads // kv_heads
    j = torch.arange(k.shape[0], device=q.device)
    hidden = (j[None, :] > last[:, None]) | (j[None, :] < first[:, None])
    out = torch.empty((lq, heads, dim), dtype=torch.float64, device=q.device)
    for h in range(kv_heads):
        kh, vh = k[:, h].double(), v[:, h].double()
        for i in range(h * group, (h + 1) * group):
            p = (q[:, i].double() @ kh.T * scale).masked_fill_(hidden, -math.inf).softmax(1)
            out[:, i] = torch.nan_to_num(p) @ vh
    return out


def _rows(cache, table_row, n, page):
    j = torch.arange(n, device=cache.device)
    slot = table_row.long()[j // page] * page + j % page
    return cache.reshape(-1, *cache.shape[2:])[slot]


def _norm_rope(x, weight, rope, positions):
    """x [T, H, D] in float64: RMS norm, weight, rotation of the halves."""
    half = x.shape[-1] // 2
    x = x / (x.square().mean(-1, keepdim=True) + _EPS).sqrt() * weight.double()
    c, n = rope.double()[positions.long()].split(half, 1)
    c, n = c[:, None], n[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * n, b * c + a * n], -1)


def _exact_prologue(s, case, slots):
    heads, kv_heads, dim = case["heads"], case["kv_heads"], case["dim"]
    rows = s["qkv"].double().reshape(s["qkv"].shape[0], heads + 2 * kv_heads, dim)
    q = _norm_rope(rows[:, :heads], s["q_weight"], s["rope"], s["positions"])
    k = _norm_rope(rows[:, heads:heads + kv_heads], s["k_weight"], s["rope"], s["positions"])
    k_cache, v_cache = s["k_cache"].double(), s["v_cache"].double()
    k_cache.reshape(-1, kv_heads, dim)[slots] = k
    v_cache.reshape(-1, kv_heads, dim)[slots] = rows[:, heads + kv_heads:]
    return q, k_cache, v_cache


def exact(case, seed):
    s = prepare(case, seed)
    kind, dim = case["kind"], case["dim"]
    if kind in ("decode", "layer"):
        lengths = _lengths(case["lo"], case["hi"], case["batch"], 1)
        window = case.get("window", -1)
        if kind == "layer":
            slots = torch.from_numpy(_slots(s["table"].cpu().numpy(), lengths, case["page"])).to(_DEVICE)
            q, k_cache, v_cache = _exact_prologue(s, case, slots)
        else:
            q, k_cache, v_cache = s["q"], s["k_cache"], s["v_cache"]
            k_cache.view(-1, case["kv_heads"], dim)[s["slots"]] = s["key"]
            v_cache.view(-1, case["kv_heads"], dim)[s["slots"]] = s["value"]
        out = []
        for i, n in enumerate(lengths.tolist()):
            first = torch.tensor([max(0, n - 1 - window) if window >= 0 else 0], device=_DEVICE)
            last = torch.tensor([n - 1], device=_DEVICE)
            out.append(_attend(q[i:i + 1], _rows(k_cache, s["table"][i], n, case["page"]),
                               _rows(v_cache, s["table"][i], n, case["page"]), first, last, s["scale"]))
        if kind == "decode":
            return torch.cat(out), k_cache, v_cache
        return torch.cat(out), q, k_cache, v_cache, _prefix_sums(lengths), slots
    if kind == "prefill":
        cu_q, cu_k, out = s["cu_q"].tolist(), s["cu_k"].tolist(), []
        for i in range(case["batch"]):
            lq, lk = cu_q[i + 1] - cu_q[i], cu_k[i + 1] - cu_k[i]
            if case["paged"]:
                k, v = (_rows(s[c], s["table"][i], lk, case["page"]) for c in ("k_cache", "v_cache"))
            else:
                k, v = s["k"][cu_k[i]:cu_k[i + 1]], s["v"][cu_k[i]:cu_k[i + 1]]
            last = torch.arange(lq, device=_DEVICE) + lk - lq
            first = last - case["window"] if case["window"] >= 0 else torch.zeros_like(last)
            out.append(_attend(s["q"][cu_q[i]:cu_q[i + 1]], k, v, first, last, s["scale"]))
        return torch.cat(out)
    if kind == "prologue":
        return _exact_prologue(s, case, s["slots"])
    k_cache, v_cache = s["k_cache"], s["v_cache"]
    for c in (k_cache, v_cache):
        c[s["pairs"][:, 1]] = c[s["pairs"][:, 0]]
    ids = s["ids"].long()
    return k_cache, v_cache, *(c[ids].reshape(-1, *c.shape[2:]) for c in (k_cache, v_cache))
