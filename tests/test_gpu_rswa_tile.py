"""The query-tiled attention kernel (head_dim 64 or 128, 512 or more (row, head) pairs,
where rswa_dispatch.hpp has the tiles faster than the rows) against the
oracle: tile and key-block edges, rows of several requests in one tile, tiles left to the row
workers, grouped heads, empty rows.

Both kernels hold everything in f32; the tolerance is that of the row kernel's
tests (1e-4 absolute on outputs of order 1)."""
import numpy as np
import pytest

import oracle as O
from test_gpu_rswa import TOL, dev_f32, dev_i32, lib, ok, ptr, rand

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


@pytest.mark.parametrize("hd,kv_heads,heads", [(128, 10, 10), (64, 2, 8), (128, 2, 6)])
@pytest.mark.parametrize("lens", [
    [260],                       # one request, 4 rows in the last tile
    [284],                       # ... and 28
    [31, 33, 64, 1, 129],        # tile boundaries inside and between requests
    [3] * 40 + [70],             # short requests: tiles of many slots
])
def test_ragged_tiles(dev, hd, kv_heads, heads, lens):
    torch = _torch()
    print(f"[rswa tile] ragged hd={hd} heads={heads}/{kv_heads} lens={lens[:6]}", flush=True)
    rng = np.random.default_rng(hd + heads + len(lens))
    cap, st, n = max(max(lens) + 5, 200), kv_heads * hd, len(lens)
    K, V = rand(rng, n, cap, kv_heads, hd), rand(rng, n, cap, kv_heads, hd)
    slots = rng.permutation(n).astype(np.int32)
    d_slots = np.concatenate([[s] * m for s, m in zip(slots, lens)]).astype(np.int32)
    d_pos = np.concatenate([np.arange(m) for m in lens]).astype(np.int32)
    total = len(d_pos)
    assert total * heads >= 512 and total * heads * cap >= 98304
    q = rand(rng, total, heads, hd)
    out = torch.full((q.size,), float("nan"), dtype=torch.float32, device=dev)
    ok(lib().uocr_hip_rswa_attention_ragged(ptr(dev_f32(q, dev)), ptr(dev_f32(K, dev)), ptr(dev_f32(V, dev)),
                                            ptr(dev_i32(d_slots, dev)), ptr(dev_i32(d_pos, dev)), total, cap, heads,
                                            kv_heads, hd, ptr(out), None))
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(total, heads * hd)
    t0 = 0
    for s, m in zip(slots, lens):
        want = O.rswa_attention(q[t0:t0 + m], K[s], V[s], m, 0, heads, kv_heads, hd, True).reshape(m, -1)
        assert np.abs(got[t0:t0 + m] - want).max() <= TOL, (s, m)
        t0 += m


def test_ragged_rows_in_any_order(dev):
    """Rows of long caches, every row another slot or position (a tile costs
    more than its rows): the row workers; and a tile that mixes both."""
    torch = _torch()
    rng = np.random.default_rng(5)
    kv_heads = heads = 10
    hd, n, cap = 128, 40, 300
    K, V = rand(rng, n, cap, kv_heads, hd), rand(rng, n, cap, kv_heads, hd)
    d_slots = np.concatenate([rng.permutation(n), [7] * 50]).astype(np.int32)
    d_pos = np.concatenate([rng.integers(0, cap, n), rng.permutation(cap)[:50]]).astype(np.int32)
    total = len(d_pos)
    q = rand(rng, total, heads, hd)
    out = torch.full((q.size,), float("nan"), dtype=torch.float32, device=dev)
    print("[rswa tile] rows in any order", flush=True)
    ok(lib().uocr_hip_rswa_attention_ragged(ptr(dev_f32(q, dev)), ptr(dev_f32(K, dev)), ptr(dev_f32(V, dev)),
                                            ptr(dev_i32(d_slots, dev)), ptr(dev_i32(d_pos, dev)), total, cap, heads,
                                            kv_heads, hd, ptr(out), None))
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(total, -1)
    for t in range(total):
        L = int(d_pos[t]) + 1
        want = O.rswa_attention(q[t:t + 1], K[d_slots[t]], V[d_slots[t]], L, 0, heads, kv_heads, hd, False).ravel()
        assert np.abs(got[t] - want).max() <= TOL, t


@pytest.mark.parametrize("seq,q_start,kv_len,causal", [(64, 936, 1000, 1), (129, 0, 129, 1), (300, 0, 33, 0),
                                                       (180, -120, 60, 1), (210, 0, 50, 1),
                                                       (220, 0, 60, 0), (252, -30, 222, 1)])  # ragged last tiles
def test_one_cache_tiles(dev, seq, q_start, kv_len, causal):
    """The query-block entry points with the length on the host and on the
    device; rows before the first key (q_start < 0) have no keys and give 0."""
    torch = _torch()
    rng = np.random.default_rng(seq + kv_len)
    kv_heads = heads = 10
    hd = 128
    assert seq * heads * kv_len >= 98304
    print(f"[rswa tile] one cache seq={seq} q_start={q_start} kv_len={kv_len} causal={causal}", flush=True)
    K, V = rand(rng, kv_len, kv_heads, hd), rand(rng, kv_len, kv_heads, hd)
    q = rand(rng, seq, heads, hd)
    lo = max(0, -q_start) if causal else 0
    want = np.zeros((seq, heads * hd), np.float32)
    want[lo:] = O.rswa_attention(q[lo:], K, V, kv_len, q_start + lo, heads, kv_heads, hd, causal).reshape(seq - lo, -1)
    kc, vc, dq = dev_f32(K, dev), dev_f32(V, dev), dev_f32(q, dev)
    for devlen in (False, True):
        out = torch.full((q.size,), float("nan"), dtype=torch.float32, device=dev)
        if devlen:
            ok(lib().uocr_hip_rswa_attention_devlen(ptr(dq), ptr(kc), ptr(vc), ptr(dev_i32([kv_len], dev)), seq,
                                                    q_start, heads, kv_heads, hd, causal, ptr(out), None))
        else:
            ok(lib().uocr_hip_rswa_attention(ptr(dq), ptr(kc), ptr(vc), kv_len, seq, q_start, heads, kv_heads, hd,
                                             causal, ptr(out), None))
        torch.cuda.synchronize()
        assert np.abs(out.cpu().numpy().reshape(seq, -1) - want).max() <= TOL, devlen


@pytest.mark.parametrize("last", [33, 57])  # a last tile of 4 rows, for the row workers, and one of 28
@pytest.mark.parametrize("hd,heads,kv_heads", [(128, 10, 10), (64, 8, 2)])
def test_keys_past_the_limit_are_not_used(dev, hd, heads, kv_heads, last):
    """Rows of the cache past each request's length hold NaN and inf: the last
    key block's tail must not reach the output (a weight of 0 times NaN would)."""
    torch = _torch()
    rng = np.random.default_rng(hd)
    lens, cap = [97, 130, last], 200
    n = len(lens)
    K, V = rand(rng, n, cap, kv_heads, hd), rand(rng, n, cap, kv_heads, hd)
    for s, m in enumerate(lens):
        K[s, m:], V[s, m:] = np.nan, np.inf
    d_slots = np.concatenate([[s] * m for s, m in enumerate(lens)]).astype(np.int32)
    d_pos = np.concatenate([np.arange(m) for m in lens]).astype(np.int32)
    total = len(d_pos)
    q = rand(rng, total, heads, hd)
    out = torch.full((q.size,), float("nan"), dtype=torch.float32, device=dev)
    print(f"[rswa tile] NaN past the limit hd={hd}", flush=True)
    ok(lib().uocr_hip_rswa_attention_ragged(ptr(dev_f32(q, dev)), ptr(dev_f32(K, dev)), ptr(dev_f32(V, dev)),
                                            ptr(dev_i32(d_slots, dev)), ptr(dev_i32(d_pos, dev)), total, cap, heads,
                                            kv_heads, hd, ptr(out), None))
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(total, heads * hd)
    t0 = 0
    for s, m in enumerate(lens):
        want = O.rswa_attention(q[t0:t0 + m], K[s, :m], V[s, :m], m, 0, heads, kv_heads, hd, True).reshape(m, -1)
        assert np.abs(got[t0:t0 + m] - want).max() <= TOL, s
        t0 += m


@pytest.mark.parametrize("last", [33, 57])  # a last tile of 4 rows, for the row workers, and one of 28
@pytest.mark.parametrize("hd,heads,kv_heads", [(128, 10, 10), (64, 8, 2)])
def test_non_finite_values_stay_with_their_rows(dev, hd, heads, kv_heads, last):
    """One request's V holds inf and NaN: the other requests' rows in the same
    tiles, and its own rows before those positions, don't see them."""
    torch = _torch()
    rng = np.random.default_rng(hd + 1)
    lens, cap = [97, 130, last], 200
    n = len(lens)
    K, V = rand(rng, n, cap, kv_heads, hd), rand(rng, n, cap, kv_heads, hd)
    V[1, 70, :, 3], V[1, 100] = np.inf, np.nan
    d_slots = np.concatenate([[s] * m for s, m in enumerate(lens)]).astype(np.int32)
    d_pos = np.concatenate([np.arange(m) for m in lens]).astype(np.int32)
    total = len(d_pos)
    q = rand(rng, total, heads, hd)
    out = torch.full((q.size,), float("nan"), dtype=torch.float32, device=dev)
    print(f"[rswa tile] inf and NaN values hd={hd}", flush=True)
    ok(lib().uocr_hip_rswa_attention_ragged(ptr(dev_f32(q, dev)), ptr(dev_f32(K, dev)), ptr(dev_f32(V, dev)),
                                            ptr(dev_i32(d_slots, dev)), ptr(dev_i32(d_pos, dev)), total, cap, heads,
                                            kv_heads, hd, ptr(out), None))
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(total, heads, hd)
    t0 = 0
    for s, m in enumerate(lens):
        clean = 70 if s == 1 else m
        want = O.rswa_attention(q[t0:t0 + clean], K[s, :clean], V[s, :clean], clean, 0, heads, kv_heads, hd,
                                True).reshape(clean, heads, hd)
        assert np.abs(got[t0:t0 + clean] - want).max() <= TOL, s
        if s == 1:
            assert not np.isfinite(got[t0 + 70:t0 + 100, :, 3]).any()
            assert not np.isfinite(got[t0 + 100:t0 + m]).any()
        t0 += m


@pytest.mark.parametrize("last", [33, 49])
@pytest.mark.parametrize("hd,heads,kv_heads", [(128, 10, 10), (64, 8, 2)])
def test_output_may_be_the_queries(dev, hd, heads, kv_heads, last):
    """out == q, with inf and NaN values in reach of some rows (whose tiles are
    partly done again): the same bits as with an output of its own."""
    torch = _torch()
    rng = np.random.default_rng(hd + 2)
    lens, cap = [197, 230, last], 300
    n = len(lens)
    K, V = rand(rng, n, cap, kv_heads, hd), rand(rng, n, cap, kv_heads, hd)
    V[1, 70, :, 3], V[1, 100], K[0, 190] = np.inf, np.nan, np.nan
    d_slots = dev_i32(np.concatenate([[s] * m for s, m in enumerate(lens)]).astype(np.int32), dev)
    d_pos = dev_i32(np.concatenate([np.arange(m) for m in lens]).astype(np.int32), dev)
    total = sum(lens)
    q = dev_f32(rand(rng, total, heads, hd), dev)
    out = torch.full_like(q, 7.0)
    kc, vc = dev_f32(K, dev), dev_f32(V, dev)
    print(f"[rswa tile] out == q hd={hd}", flush=True)
    for dst in (out, q):
        ok(lib().uocr_hip_rswa_attention_ragged(ptr(q), ptr(kc), ptr(vc), ptr(d_slots), ptr(d_pos), total, cap, heads,
                                                kv_heads, hd, ptr(dst), None))
    torch.cuda.synchronize()
    a, b = out.cpu().numpy(), q.cpu().numpy()
    assert np.array_equal(a, b, equal_nan=True)
    assert not np.isfinite(a).all() and np.isfinite(a).mean() > 0.5


def _rows_want(q, K, V, slots, pos, heads, kv_heads, hd):
    """Attention of every row over its slot's rows [0, pos], in 64 bits."""
    T, cap = len(slots), K.shape[1]
    q = q.reshape(T, heads, hd).astype(np.float64)
    out = np.empty_like(q)
    dead = np.arange(cap)[None] > pos[:, None]
    for h in range(heads):
        g = h // (heads // kv_heads)
        s = np.einsum("td,tcd->tc", q[:, h], K[slots, :, g].astype(np.float64)) / np.sqrt(hd)
        s[dead] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = np.einsum("tc,tcd->td", p / p.sum(1, keepdims=True), V[slots, :, g].astype(np.float64))
    return out.reshape(T, -1)


@pytest.mark.parametrize("hd,heads,kv_heads", [(128, 10, 10), (64, 8, 2), (128, 32, 8), (64, 32, 8)])
@pytest.mark.parametrize("name,lens,starts", [
    ("a long end", [129, 95, 65, 97, 80], 0),  # a tile with its last row: 32 heads fill the chip and keep it a tile
    ("one row each", [1] * 203, "any"),                        # row workers only, more than one row each
    ("4 rows each", [4] * 60, 0), ("5 rows each", [5] * 45, 7),  # many passes: left to the workers
    ("20 rows each at 130", [20] * 6, 130),                    # long keys, two or three requests in a tile: left to the workers
    ("52 rows at 100", [52, 53], 100),
    ("20 rows each", [20] * 14, 0),                            # few passes: tiles, a short last one
    ("mixed", [1] * 70 + [130, 1, 9, 64, 2], "any"),           # both kinds in one call
])
def test_tiles_and_row_workers(dev, hd, heads, kv_heads, name, lens, starts):
    """Every row is taken once, by a tile or by a worker, whatever the mix of requests."""
    torch = _torch()
    rng = np.random.default_rng(len(lens) + hd)
    cap, n = 160, len(lens)
    K, V = rand(rng, n, cap, kv_heads, hd), rand(rng, n, cap, kv_heads, hd)
    first = [int(rng.integers(0, cap - m + 1)) if starts == "any" else starts for m in lens]
    slots = np.concatenate([[s] * m for s, m in zip(rng.permutation(n), lens)]).astype(np.int32)
    pos = np.concatenate([f + np.arange(m) for f, m in zip(first, lens)]).astype(np.int32)
    total = len(pos)
    q = rand(rng, total, heads, hd)
    out = torch.full((q.size,), float("nan"), dtype=torch.float32, device=dev)
    print(f"[rswa tile] {name} hd={hd}", flush=True)
    ok(lib().uocr_hip_rswa_attention_ragged(ptr(dev_f32(q, dev)), ptr(dev_f32(K, dev)), ptr(dev_f32(V, dev)),
                                            ptr(dev_i32(slots, dev)), ptr(dev_i32(pos, dev)), total, cap, heads,
                                            kv_heads, hd, ptr(out), None))
    torch.cuda.synchronize()
    want = _rows_want(q, K, V, slots, pos, heads, kv_heads, hd)
    assert np.abs(out.cpu().numpy().reshape(total, -1) - want).max() <= TOL


def test_row_workers_past_256_tiles(dev):
    """A call of more tiles than a worker looks at at once."""
    torch = _torch()
    rng = np.random.default_rng(8)
    hd, heads, kv_heads, cap, total = 64, 2, 1, 5, 32 * 256 + 77
    K, V = rand(rng, total, cap, kv_heads, hd), rand(rng, total, cap, kv_heads, hd)
    slots = rng.permutation(total).astype(np.int32)
    pos = rng.integers(0, cap, total).astype(np.int32)
    q = rand(rng, total, heads, hd)
    out = torch.full((q.size,), float("nan"), dtype=torch.float32, device=dev)
    print("[rswa tile] past 256 tiles", flush=True)
    ok(lib().uocr_hip_rswa_attention_ragged(ptr(dev_f32(q, dev)), ptr(dev_f32(K, dev)), ptr(dev_f32(V, dev)),
                                            ptr(dev_i32(slots, dev)), ptr(dev_i32(pos, dev)), total, cap, heads,
                                            kv_heads, hd, ptr(out), None))
    torch.cuda.synchronize()
    want = _rows_want(q, K, V, slots, pos, heads, kv_heads, hd)
    assert np.abs(out.cpu().numpy().reshape(total, -1) - want).max() <= TOL
