"""GPU parity of prefill attention (paged and contiguous, causal, GQA, window) against
the oracle.

Tolerance (the target's, for bf16/f16 output vs an fp32-accumulated reference):
max-abs 2e-2 and max-rel 1e-2 (helpers.assert_attn_close).  The oracle's prefill
(oracle/oxide_oracle.c) is pinned in tests/test_oracle.py against a dense numpy fp64
routine, the decode oracle row by row, and a hand-worked FlashAttention 2 mask case.
"""
import math

import numpy as np
import pytest

import oracle
from helpers import assert_attn_close, normal_bits, to_f32, to_torch

pytestmark = pytest.mark.gpu


def _case(seed, lq, lk, Hq, Hkv, D, BS, dtype="bf16", spare=2):
    rng = np.random.default_rng(seed)
    lq = np.asarray(lq, np.int64)
    lk = np.asarray(lk, np.int64)
    B = len(lq)
    nblk = (lk + BS - 1) // BS
    NB = int(nblk.sum()) + spare
    perm = rng.permutation(NB).astype(np.int32)
    table = np.zeros((B, max(int(nblk.max()), 1)), np.int32)
    pos = 0
    for b in range(B):
        table[b, :nblk[b]] = perm[pos:pos + nblk[b]]
        pos += nblk[b]
    cuq = np.zeros(B + 1, np.uint32)
    cuq[1:] = np.cumsum(lq)
    cuk = np.zeros(B + 1, np.uint32)
    cuk[1:] = np.cumsum(lk)
    q = normal_bits(rng, (int(cuq[-1]), Hq, D), dtype)
    kc = normal_bits(rng, (NB, BS, Hkv, D), dtype)
    vc = normal_bits(rng, (NB, BS, Hkv, D), dtype)
    return q, kc, vc, cuq, cuk, table


def _contiguous(kc, cuk, table):
    NB, BS, Hkv, D = kc.shape
    rows = []
    for b in range(len(cuk) - 1):
        j = np.arange(int(cuk[b + 1] - cuk[b]))
        rows.append(table[b, j // BS].astype(np.int64) * BS + j % BS)
    rows = np.concatenate(rows) if rows else np.zeros(0, np.int64)
    return np.ascontiguousarray(kc.reshape(-1, Hkv, D)[rows])


def _gpu(device, q, k, v, cuq, cuk, table, scale, window, dtype, paged=True):
    import torch
    import oxide_paged_kv as ox

    t = lambda a: to_torch(a, dtype, device)  # noqa: E731
    mq = int(np.max(np.diff(cuq))) if len(cuq) > 1 else 0
    mk = int(np.max(np.diff(cuk))) if len(cuk) > 1 else 0
    out = ox.prefill_attn(t(q), t(k), t(v), torch.from_numpy(cuq.view(np.int32)).to(device),
                          torch.from_numpy(cuk.view(np.int32)).to(device), mq, mk, scale,
                          torch.from_numpy(table).to(device) if paged else None,
                          None if window < 0 else window)
    torch.cuda.synchronize()
    return out


CASES = [
    # (lq, lk, Hq, Hkv, D, BS, window, dtype)
    ([300, 77], [300, 77], 32, 8, 128, 256, -1, "bf16"),              # plain prompts, G=4
    ([128, 40, 200], [1000, 40, 457], 32, 8, 128, 256, -1, "bf16"),   # prefix hits (Lk > Lq)
    ([64, 9], [64, 4], 16, 8, 128, 16, -1, "bf16"),                   # Lk < Lq: leading rows see nothing
    ([0, 50, 0, 1], [10, 50, 0, 1], 16, 8, 128, 256, -1, "bf16"),     # empty query lists / keys
    ([513, 100], [513, 900], 16, 8, 128, 256, 100, "bf16"),           # window 100
    ([200], [1200], 64, 8, 128, 256, 4096, "bf16"),                   # G=8, window > context
    ([130, 70], [130, 270], 8, 8, 128, 32, -1, "f16"),                # G=1, f16, BS=32
    ([100, 33], [100, 66], 4, 2, 64, 16, 7, "bf16"),                  # G=2, D=64, window 7
    ([90], [300], 32, 2, 64, 256, -1, "f16"),                         # G=16, D=64
    ([40], [40], 24, 8, 128, 256, -1, "bf16"),                        # G=3 (rows not a power of 2)
    # No cached prefix and prompts of at most 2048 tokens: workgroups take row tiles in
    # pairs (n - 1 - i, then i), including an odd tile count's middle tile alone.
    ([70, 33], [70, 33], 32, 8, 128, 256, -1, "bf16"),                # 3 and 2 row tiles
    ([300, 150], [300, 150], 32, 8, 128, 64, 50, "f16"),              # window 50, BS=64
    ([2048], [2048], 16, 8, 64, 32, -1, "bf16"),                      # the longest paired prompt
]


@pytest.mark.parametrize("case", CASES, ids=[f"c{i}" for i in range(len(CASES))])
def test_prefill_paged_vs_oracle(device, case):
    lq, lk, Hq, Hkv, D, BS, window, dtype = case
    q, kc, vc, cuq, cuk, table = _case(21, lq, lk, Hq, Hkv, D, BS, dtype)
    scale = 1.0 / math.sqrt(D)
    print(f"prefill case lq={lq} lk={lk} Hq={Hq} Hkv={Hkv} D={D} BS={BS} w={window} {dtype}", flush=True)
    got = to_f32(_gpu(device, q, kc, vc, cuq, cuk, table, scale, window, dtype))
    want = oracle.prefill_attention(q, kc, vc, cuq, cuk, scale, table, window, dtype)
    assert_attn_close(got, want)
    # Rows that see no key are exactly zero.
    for b in range(len(lq)):
        for i in range(lq[b]):
            if i + lk[b] - lq[b] < 0:
                assert not got[int(cuq[b]) + i].any()


def _random_shapes(seed, n):
    """Seeded random shapes: 1-3 prompts of up to 300 new tokens behind up to 500
    cached keys (or fewer keys than queries), kv heads 1/2/4/8, groups 1-8 and 16,
    D 64/128, page sizes 16/32/64/256 (per-row and per-tile block lookups), windows,
    bf16/f16; at most ~1e9 multiply-adds per case for the oracle."""
    rng = np.random.default_rng(seed)
    out = []
    while len(out) < n:
        B = int(rng.integers(1, 4))
        Hkv = int(rng.choice([1, 2, 4, 8]))
        G = int(rng.choice([1, 2, 3, 4, 5, 6, 7, 8, 16]))
        D = int(rng.choice([64, 128]))
        lq = rng.integers(0, 301, B)
        pre = rng.integers(0, 501, B) if rng.random() < 0.7 else -rng.integers(0, 50, B)
        lk = np.maximum(lq + pre, 0)
        if lq.sum() == 0 or lk.sum() == 0:
            continue
        if int((lq * lk).sum()) * G * Hkv * D > 1e9:
            continue
        window = -1 if rng.random() < 0.6 else int(rng.integers(0, 600))
        out.append((lq.tolist(), lk.tolist(), G * Hkv, Hkv, D, int(rng.choice([16, 32, 64, 256])), window,
                    str(rng.choice(["bf16", "f16"]))))
    return out


@pytest.mark.parametrize("case", _random_shapes(77, 24), ids=[f"r{i}" for i in range(24)])
def test_prefill_random_shapes_vs_oracle(device, case):
    lq, lk, Hq, Hkv, D, BS, window, dtype = case
    q, kc, vc, cuq, cuk, table = _case(31, lq, lk, Hq, Hkv, D, BS, dtype)
    scale = 1.0 / math.sqrt(D)
    print(f"prefill random lq={lq} lk={lk} Hq={Hq} Hkv={Hkv} D={D} BS={BS} w={window} {dtype}", flush=True)
    got = to_f32(_gpu(device, q, kc, vc, cuq, cuk, table, scale, window, dtype))
    assert_attn_close(got, oracle.prefill_attention(q, kc, vc, cuq, cuk, scale, table, window, dtype))


# 32 prompts of about one length fill four rounds of the chip's workgroup slots, so that
# row tiles go in pairs (9 tiles, the middle one alone; shorter prompts of 8); a ragged
# batch of the same grid takes them one by one.
@pytest.mark.parametrize("lens", [[288, 257, 256, 225] * 8, [288, 1, 33, 0] * 8], ids=["pairs", "ragged"])
def test_prefill_many_prompts_vs_oracle(device, lens):
    q, kc, vc, cuq, cuk, table = _case(61, lens, lens, 32, 8, 64, 256)
    got = to_f32(_gpu(device, q, kc, vc, cuq, cuk, table, 0.125, -1, "bf16"))
    assert_attn_close(got, oracle.prefill_attention(q, kc, vc, cuq, cuk, 0.125, table, -1, "bf16"))


# (sequence, kv head) units that do not fill the 8 XCDs evenly: their row tiles alternate
# over 8, 2 (12 units; tile counts 7 and 1), 4 and 8 (10 and 9 units) XCDs.
UNEVEN = [
    # (lq, Hq, Hkv, D, BS, window, dtype)
    ([300], 8, 1, 128, 64, -1, "bf16"),
    ([100, 1, 113], 28, 4, 128, 256, -1, "f16"),
    ([70, 5, 64, 33, 129], 8, 2, 64, 16, 50, "bf16"),
    ([40] * 9, 16, 1, 64, 256, -1, "bf16"),
]


@pytest.mark.parametrize("case", UNEVEN, ids=[f"u{i}" for i in range(len(UNEVEN))])
def test_prefill_uneven_units_vs_oracle(device, case):
    lens, Hq, Hkv, D, BS, window, dtype = case
    q, kc, vc, cuq, cuk, table = _case(71, lens, lens, Hq, Hkv, D, BS, dtype)
    scale = 1.0 / math.sqrt(D)
    print(f"prefill uneven units lq={lens} Hq={Hq} Hkv={Hkv} D={D} BS={BS} w={window} {dtype}", flush=True)
    got = to_f32(_gpu(device, q, kc, vc, cuq, cuk, table, scale, window, dtype))
    assert_attn_close(got, oracle.prefill_attention(q, kc, vc, cuq, cuk, scale, table, window, dtype))


# Queries behind long cached contexts, whose keys are split over workgroups: the piece
# and tile edges, sequences with nothing to split or no queries, the smallest batch and
# the largest that is split (64), rows of 128 that groups of 7 and 5 do not fill.
BALANCED = [
    # (lq, lk, Hq, Hkv, D, BS, window, dtype)
    ([1], [1500], 32, 8, 128, 256, -1, "bf16"),                       # one row tile, pieces of 8 steps
    ([33, 1], [1025, 1600], 32, 8, 128, 64, -1, "f16"),               # one row past a row tile
    ([40, 0, 70, 12], [2100, 900, 1000, 12], 28, 4, 128, 256, -1, "bf16"),  # G=7; no queries; no cached keys
    ([30, 18], [1400, 5], 40, 8, 64, 16, -1, "bf16"),                 # Lk < Lq beside a split one; per-row pages
    ([64, 64], [3000, 1900], 16, 8, 128, 256, 1000, "f16"),           # window over several pieces
    ([1] * 63 + [9], [600 + 31 * i for i in range(64)], 16, 2, 64, 32, -1, "bf16"),  # 64 sequences
]


@pytest.mark.parametrize("case", BALANCED, ids=[f"b{i}" for i in range(len(BALANCED))])
def test_prefill_behind_long_context_vs_oracle(device, case):
    from oxide_paged_kv import _lib

    lq, lk, Hq, Hkv, D, BS, window, dtype = case
    assert _lib.load().prefill_attention_workspace_size(len(lq), Hq, Hkv, D, max(lq), max(lk), window) > 0
    q, kc, vc, cuq, cuk, table = _case(51, lq, lk, Hq, Hkv, D, BS, dtype)
    scale = 1.0 / math.sqrt(D)
    print(f"prefill balanced lq={lq[:4]} lk={lk[:4]} Hq={Hq} Hkv={Hkv} D={D} BS={BS} w={window} {dtype}", flush=True)
    got = to_f32(_gpu(device, q, kc, vc, cuq, cuk, table, scale, window, dtype))
    assert_attn_close(got, oracle.prefill_attention(q, kc, vc, cuq, cuk, scale, table, window, dtype))


@pytest.mark.parametrize("case", [CASES[1], CASES[4], CASES[7]], ids=["prefix", "window", "d64"])
def test_prefill_contiguous_equals_paged(device, case):
    """flash_attn_varlen form (contiguous K/V): same kernel, so bit-identical to the paged
    form over the same keys, and within tolerance of the oracle."""
    import torch

    lq, lk, Hq, Hkv, D, BS, window, dtype = case
    q, kc, vc, cuq, cuk, table = _case(22, lq, lk, Hq, Hkv, D, BS, dtype)
    kcont, vcont = _contiguous(kc, cuk, table), _contiguous(vc, cuk, table)
    print(f"prefill contiguous lq={lq} lk={lk} D={D} w={window}", flush=True)
    paged = _gpu(device, q, kc, vc, cuq, cuk, table, 0.1, window, dtype)
    cont = _gpu(device, q, kcont, vcont, cuq, cuk, table, 0.1, window, dtype, paged=False)
    assert torch.equal(paged, cont)
    want = oracle.prefill_attention(q, kcont, vcont, cuq, cuk, 0.1, None, window, dtype)
    assert_attn_close(to_f32(cont), want)


def test_prefill_placement_invariance(device):
    """Moving blocks to other physical ids (same logical content) changes nothing, bit for bit."""
    import torch

    lq, lk = [100, 60], [700, 60]
    q, kc, vc, cuq, cuk, table = _case(23, lq, lk, 32, 8, 128, 16, "bf16", spare=30)
    NB = kc.shape[0]
    perm = np.random.default_rng(5).permutation(NB).astype(np.int32)
    kc2 = np.empty_like(kc)
    vc2 = np.empty_like(vc)
    kc2[perm] = kc
    vc2[perm] = vc
    table2 = perm[table]
    a = _gpu(device, q, kc, vc, cuq, cuk, table, 0.08, -1, "bf16")
    b = _gpu(device, q, kc2, vc2, cuq, cuk, table2, 0.08, -1, "bf16")
    assert torch.equal(a, b)


def test_prefill_long_prompt_rows_vs_decode_oracle(device):
    """Two 4096-token prompts behind a 1000-token prefix (Qwen3-8B heads): sampled rows
    checked against the decode oracle over each row's causal prefix."""
    lq, lk = [4096, 2500], [5096, 2500]
    q, kc, vc, cuq, cuk, table = _case(24, lq, lk, 32, 8, 128, 256, "bf16")
    scale = 1 / math.sqrt(128)
    print("prefill long prompt 4096+2500", flush=True)
    got = to_f32(_gpu(device, q, kc, vc, cuq, cuk, table, scale, -1, "bf16"))
    rng = np.random.default_rng(0)
    for b in range(2):
        for i in np.concatenate([[0, lq[b] - 1], rng.integers(0, lq[b], 6)]):
            L = int(i) + lk[b] - lq[b] + 1
            t = int(cuq[b]) + int(i)
            want = oracle.paged_decode_attention(q[t][None], kc, vc, np.array([0, L], np.uint32),
                                                 table[b][None], scale, -1, "bf16")
            assert_attn_close(got[t][None], want)


def test_prefill_rejects_bad_arguments(device):
    import torch
    import oxide_paged_kv as ox

    q = torch.zeros((4, 8, 96), dtype=torch.bfloat16, device=device)  # head_dim 96: not built
    cu = torch.tensor([0, 4], dtype=torch.int32, device=device)
    with pytest.raises(ox.OxideError):
        ox.prefill_attn(q, q, q, cu, cu, 4, 4, 1.0)
    q = torch.zeros((4, 8, 128), dtype=torch.float32, device=device)  # f32: not supported
    with pytest.raises(ox.OxideError):
        ox.prefill_attn(q, q, q, cu, cu, 4, 4, 1.0)


@pytest.mark.parametrize("window", [-1, 300])
def test_prefill_last_rows_equal_decode(device, window):
    """Cross-kernel invariant: the last query row of every prompt sees exactly the keys a
    decode step over the same cache sees, so the two kernels agree (within the
    attention tolerance: different accumulation orders)."""
    import torch
    import oxide_paged_kv as ox
    from helpers import assert_attn_close

    lq, lk = [200, 77, 1, 513], [1200, 77, 40, 513]
    q, kc, vc, cuq, cuk, table = _case(25, lq, lk, 32, 8, 128, 256, "bf16")
    pre = to_f32(_gpu(device, q, kc, vc, cuq, cuk, table, 0.09, window, "bf16"))
    last = np.array([int(cuq[b + 1]) - 1 for b in range(len(lq))])
    dec = ox.decode_attn(to_torch(q[last], "bf16", device), to_torch(kc, "bf16", device),
                         to_torch(vc, "bf16", device), torch.from_numpy(cuk.view(np.int32)).to(device),
                         torch.from_numpy(table).to(device), max(lk), 0.09, None if window < 0 else window)
    torch.cuda.synchronize()
    assert_attn_close(pre[last], to_f32(dec))


# An infinite or NaN V reaches only rows whose wave (32 rows) sees some key of its 64-key
# tile.  Group 1: a wave is 32 tokens, a workgroup 128.  (window, cached, bad key, the
# tokens of waves that see nothing of the key's tile)
BAD_V = [
    (-1, 0, 200, (0, 192)),      # keys of tile 192..255 are after every token below 192
    (20, 0, 70, (160, 256)),     # window 20: tokens from 160 on see keys from 140 on
    (-1, 4096, 200, (0, 192)),   # the same behind a cached context, keys split over workgroups
    (20, 4096, 70, (160, 256)),
]


@pytest.mark.parametrize("case", BAD_V, ids=["causal", "window", "causal-cached", "window-cached"])
@pytest.mark.parametrize("BS", [64, 16])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_prefill_bad_values_stay_in_their_tile(device, case, BS, bad):
    window, cached, key, (lo, hi) = case
    q, kc, vc, cuq, cuk, table = _case(81, [256], [256 + cached], 1, 1, 64, BS)
    print(f"prefill bad V window={window} cached={cached} BS={BS} {bad}", flush=True)
    clean = to_f32(_gpu(device, q, kc, vc, cuq, cuk, table, 0.125, window, "bf16"))
    vb = vc.copy()
    j = cached + key
    vb[table[0, j // BS], j % BS] = oracle.f32_to_bf16_bits(np.full((1, 64), bad, np.float32))
    got = to_f32(_gpu(device, q, kc, vb, cuq, cuk, table, 0.125, window, "bf16"))
    assert not np.isfinite(got[key]).any()  # the token itself sees the key
    assert np.array_equal(got[lo:hi], clean[lo:hi])


def _entry(device, q, k, v, cuq, cuk, table, scale, window, dtype, workspace_bytes=None, offset=0):
    """The C entries: paged_prefill_attention, or with workspace_bytes the workspace form
    over that many bytes from `offset` of a guarded buffer (0 = no workspace).  Returns
    the output and whether the bytes outside the stated workspace are as they were."""
    import torch
    from oxide_paged_kv import _lib

    L = _lib.load()
    t = lambda a: to_torch(a, dtype, device)  # noqa: E731
    i32 = lambda a: torch.from_numpy(a.view(np.int32)).to(device)  # noqa: E731
    qd, kd, vd, cq, ck, tb = t(q), t(k), t(v), i32(cuq), i32(cuk), i32(table)
    out = torch.zeros_like(qd)
    (_, Hq, D), (NB, BS, Hkv, _) = q.shape, k.shape
    args = [out, qd, kd, vd, cq, ck, tb]
    sizes = [table.shape[1], NB, len(cuq) - 1, Hq, Hkv, D, BS, int(np.max(np.diff(cuq))), int(np.max(np.diff(cuk))),
             window, scale]
    code, stream = _lib.DTYPE_BF16 if dtype == "bf16" else _lib.DTYPE_F16, torch.cuda.current_stream().cuda_stream
    guard = torch.full(((workspace_bytes or 0) + 8192,), 0x5A, dtype=torch.uint8, device=device)
    ptrs = [a.data_ptr() for a in args]
    if workspace_bytes is None:
        L.paged_prefill_attention(*ptrs, *sizes, code, stream)
    else:
        L.paged_prefill_attention_workspace(*ptrs, *sizes, guard.data_ptr() + offset if workspace_bytes else None,
                                            workspace_bytes, code, stream)
    _lib.check()
    torch.cuda.synchronize()
    return out, bool((guard[:offset] == 0x5A).all()) and bool((guard[offset + (workspace_bytes or 0):] == 0x5A).all())


def _workspace_size(q, k, cuq, cuk, window):
    from oxide_paged_kv import _lib

    return int(_lib.load().prefill_attention_workspace_size(
        len(cuq) - 1, q.shape[1], k.shape[2], q.shape[2], int(np.max(np.diff(cuq))), int(np.max(np.diff(cuk))), window))


@pytest.mark.parametrize("lk", [1500, 2600])  # three and six pieces of a row tile
@pytest.mark.parametrize("what", ["q nan", "q inf", "k nan", "v inf last", "v inf first", "v nan"])
def test_prefill_split_keys_pass_nan_and_infinity(device, lk, what):
    """NaN and infinities come out of keys split over workgroups as from the plain entry."""
    q, kc, vc, cuq, cuk, table = _case(83, [3], [lk], 8, 2, 64, 64)
    bits = lambda x: oracle.f32_to_bf16_bits(np.full((), x, np.float32))  # noqa: E731
    at = lambda j: (table[0, j // 64], j % 64)  # noqa: E731
    if what[0] == "q":
        q[1] = bits(np.nan if "nan" in what else np.inf)
    elif what[0] == "k":
        kc[at(700)] = bits(np.nan)
    else:
        vc[at(3 if "first" in what else lk - 10)] = bits(np.nan if "nan" in what else np.inf)
    need = _workspace_size(q, kc, cuq, cuk, -1)
    assert need > 0
    print(f"prefill split lk={lk} {what}", flush=True)
    want = to_f32(_entry(device, q, kc, vc, cuq, cuk, table, 0.125, -1, "bf16")[0])
    got = to_f32(_entry(device, q, kc, vc, cuq, cuk, table, 0.125, -1, "bf16", need)[0])
    assert not np.isfinite(want).all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    fin = np.isfinite(want)
    assert np.array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)]))
    assert_attn_close(got[fin], want[fin])


# The balanced launch on the real lengths: (lq, lk, whether tiles are cut).  16 query heads
# on one kv head (8 tokens per row tile), 256 CUs with two slots each.
REAL_LENGTHS = [
    ([256] * 8, [4096] * 8, False),                               # 256 tiles of one length
    ([128] * 28, [7600 + 21 * i for i in range(28)], False),      # 448 tiles of about one length
    ([128] * 40, [3328 + 28 * i for i in range(40)], False),      # 640 tiles: more than slots
    ([256] * 8, [1024 + 438 * i for i in range(8)], True),        # 256 ragged ones
    ([128] * 40, [500] * 39 + [12000], True),                     # 640, one sequence far longer
    ([1024], [8704], True),                                       # pieces in one round
    ([704, 1024], [12288, 18432], True),                          # and in two (a third of it: as long whole)
]


@pytest.mark.parametrize("case", REAL_LENGTHS, ids=[f"r{i}" for i in range(len(REAL_LENGTHS))])
def test_prefill_cuts_tiles_where_the_lengths_call_for_it(device, case):
    """Where whole tiles take no longer the workspace entry is the plain one, bit for bit;
    elsewhere it differs by rounding only."""
    import torch

    lq, lk, cut = case
    if torch.cuda.get_device_properties(device).multi_processor_count != 256:
        pytest.skip("the sizes are for 256 CUs")
    q, kc, vc, cuq, cuk, table = _case(85, lq, lk, 16, 1, 128, 256)
    need = _workspace_size(q, kc, cuq, cuk, -1)
    assert need > 0
    print(f"prefill real lengths lq={lq[:2]} lk={lk[:2]}", flush=True)
    want, _ = _entry(device, q, kc, vc, cuq, cuk, table, 0.09, -1, "bf16")
    got, _ = _entry(device, q, kc, vc, cuq, cuk, table, 0.09, -1, "bf16", need)
    again, _ = _entry(device, q, kc, vc, cuq, cuk, table, 0.09, -1, "bf16", need)
    assert torch.equal(got, again)
    assert torch.equal(got, want) != cut
    assert_attn_close(to_f32(got), to_f32(want))


@pytest.mark.parametrize("case", [BALANCED[2], BALANCED[4]], ids=["b2", "b4"])
def test_prefill_workspace_forms(device, case):
    """No workspace, a misaligned one and one a byte short are the plain call; the full one
    is not written past its end.  The plain entries against the oracle too."""
    import torch
    from oxide_paged_kv import _lib

    lq, lk, Hq, Hkv, D, BS, window, dtype = case
    q, kc, vc, cuq, cuk, table = _case(87, lq, lk, Hq, Hkv, D, BS, dtype)
    scale = 1.0 / math.sqrt(D)
    need = _workspace_size(q, kc, cuq, cuk, window)
    assert need > 0
    print(f"prefill workspace forms lq={lq} lk={lk} window={window} {dtype}", flush=True)
    args = (device, q, kc, vc, cuq, cuk, table, scale, window, dtype)
    plain, _ = _entry(*args)
    want = oracle.prefill_attention(q, kc, vc, cuq, cuk, scale, table, window, dtype)
    assert_attn_close(to_f32(plain), want)
    for size, offset in ((0, 0), (need, 4), (need - 1, 0)):
        got, kept = _entry(*args, size, offset)
        assert torch.equal(got, plain) and kept
    got, kept = _entry(*args, need, 256)
    assert kept and not torch.equal(got, plain)  # keys were split
    assert_attn_close(to_f32(got), want)

    # Contiguous K/V: the plain entry, and the workspace entry without one.
    L = _lib.load()
    t = lambda a: to_torch(a, dtype, device)  # noqa: E731
    i32 = lambda a: torch.from_numpy(a.view(np.int32)).to(device)  # noqa: E731
    qd, kd, vd, cq, ck = t(q), t(_contiguous(kc, cuk, table)), t(_contiguous(vc, cuk, table)), i32(cuq), i32(cuk)
    code, stream = _lib.DTYPE_BF16 if dtype == "bf16" else _lib.DTYPE_F16, torch.cuda.current_stream().cuda_stream
    for name, ws in (("varlen_prefill_attention", ()), ("varlen_prefill_attention_workspace", (None, 0))):
        out = torch.zeros_like(qd)
        getattr(L, name)(out.data_ptr(), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), cq.data_ptr(), ck.data_ptr(),
                         kd.shape[0], len(lq), Hq, Hkv, D, max(lq), max(lk), window, scale, *ws, code, stream)
        _lib.check()
        torch.cuda.synchronize()
        assert torch.equal(out, plain)
