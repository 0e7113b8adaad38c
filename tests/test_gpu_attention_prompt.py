"""The prompt attention kernel (split-f16 matrix products) on its own: tile
and block edges, value ranges its scales have to follow, values that are not
finite, and the rule that chooses it.  Parity against the oracle
(models/src/transformer.rs:301-374).

Bar: 2e-5 of the largest |V| of the same output dim.  Outputs are convex
combinations of V rows, and a score is a dot product of 64 or 128 terms, each
to 2^-22 of its |q||k| (two values split to 2^-23 each, their small parts'
product left out), so at the sizes here (|score| below 10) a weight is off by
less than 10 * 2^-21 and an output by less than 1e-5 of the largest |V|.
"""
import os

import numpy as np
import pytest

import barq_rocm as B
from barq_rocm import attention as A

pytestmark = pytest.mark.gpu
F32 = np.float32


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def backend(min_q):
    old = os.environ.get("BARQ_ATTN_MFMA_MIN_Q")
    os.environ["BARQ_ATTN_MFMA_MIN_Q"] = str(min_q)
    try:
        return B.Backend(0)
    finally:
        if old is None:
            os.environ.pop("BARQ_ATTN_MFMA_MIN_Q", None)
        else:
            os.environ["BARQ_ATTN_MFMA_MIN_Q"] = old


@pytest.fixture(scope="module")
def prompt_be(be):
    b = backend(1)
    yield b
    b.close()


def attend(b, q, k, v, start, n_head):
    n_kv, kv_len, hd = k.shape
    q_len = q.shape[1]
    c = A.KVCache(b, kv_len, 1, n_kv, hd)
    c.append(0, k, v, kv_len, hd, mem=B.MEM_HOST)
    out = A.compute_attention(b, dev(q), c, 0, n_head, n_kv, hd, q_len, kv_len, start).cpu().numpy()
    q8 = A.compute_attention_q8k(b, dev(q), c, 0, n_head, n_kv, hd, q_len, kv_len, start).cpu().numpy()
    assert np.array_equal(q8.reshape(-1), b.quantize_act(B.Q8_K, dev(out.reshape(q_len, -1))).cpu().numpy().reshape(-1))
    c.close()
    return out


def close(out, ref, v, n_head):
    """out, ref [q_len, n_head, hd]; v [n_kv, kv_len, hd]"""
    n_kv = v.shape[0]
    for h in range(n_head):
        top = np.max(np.abs(v[h * n_kv // n_head]), axis=0)
        err = np.abs(out[:, h] - ref[:, h])
        assert np.all(err <= 2e-5 * top + 1e-37), (h, float(np.max(err / (top + 1e-37))))


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("n_head,n_kv,q_len,start,kv_len", [
    (4, 4, 127, 0, 127),      # one query head per kv head: a tile of 128 queries, one short
    (4, 4, 129, 31, 160),     # one row into the second tile
    (8, 2, 32, 0, 32),        # exactly one tile, one block
    (8, 2, 33, 1, 34),        # a tile and a row, a block and two positions
    (12, 4, 50, 70, 120),     # three query heads per kv head: tiles cut a query's heads apart
    (8, 4, 65, 0, 70),        # positions that no query sees
    (6, 4, 40, 9, 49),        # heads that do not divide
    (16, 2, 90, 600, 690),    # pieces of every tile
])
def test_tile_edges(prompt_be, orc, hd, n_head, n_kv, q_len, start, kv_len):
    if n_head * hd % 256:
        n_head, n_kv = 2 * n_head, 2 * n_kv
    r = np.random.default_rng(hd + q_len)
    q, k, v = (r.standard_normal(s).astype(F32) for s in ((n_head, q_len, hd), (n_kv, kv_len, hd), (n_kv, kv_len, hd)))
    print("prompt attention", hd, n_head, n_kv, q_len, start, kv_len, flush=True)
    close(attend(prompt_be, q, k, v, start, n_head), orc.attention(q, k, v, n_head, q_len, kv_len, start), v, n_head)


@pytest.mark.parametrize("hd", [64, 128])
def test_value_ranges(prompt_be, orc, hd):
    """Scales per position (K), per query row (Q) and per dim (V, growing with
    the positions by up to 2^20, one dim zero for two blocks, one zero
    throughout)."""
    n_head, n_kv, q_len, kv_len = 8, 2, 100, 200
    r = np.random.default_rng(hd)
    q, k, v = (r.standard_normal(s) for s in ((n_head, q_len, hd), (n_kv, kv_len, hd), (n_kv, kv_len, hd)))
    q *= 2.0 ** r.integers(-2, 2, (n_head, q_len, 1)) * 1e12
    k *= 2.0 ** r.integers(-6, 1, (n_kv, kv_len, 1)) * 1e-12
    v *= 2.0 ** np.linspace(-100, 100, hd) * 2.0 ** (np.arange(kv_len)[:, None] // 20 * r.integers(0, 3, hd))
    v[:, :64, 3] = 0
    v[:, :, 5] = 0
    q, k, v = q.astype(F32), k.astype(F32), v.astype(F32)
    out = attend(prompt_be, q, k, v, kv_len - q_len, n_head)
    # the bar per row uses V up to it (test_values_beside_a_large_one: what it does not see)
    ref = orc.attention(q, k, v, n_head, q_len, kv_len, kv_len - q_len)
    for i in (0, 40, q_len - 1):
        close(out[i:i + 1], ref[i:i + 1], v[:, :kv_len - q_len + i + 1], n_head)


@pytest.mark.parametrize("hd", [64, 128])
def test_values_that_are_not_finite(prompt_be, orc, hd):
    """An infinity in V reaches its dim only, NaN in a key every query that
    sees it; everything else is as if they were not there."""
    n_head, n_kv, q_len, kv_len = 8, 2, 70, 70
    r = np.random.default_rng(7)
    q, k, v = (r.standard_normal(s).astype(F32) for s in ((n_head, q_len, hd), (n_kv, kv_len, hd), (n_kv, kv_len, hd)))
    v[0, 0, 9] = np.inf
    out = attend_f32(prompt_be, q, k, v, n_head)
    assert np.all(np.isposinf(out[:, :4, 9]))
    v0 = v.copy()
    v0[0, 0, 9] = 0
    ref = orc.attention(q, k, v0, n_head, q_len, kv_len, 0)
    keep = np.ones(hd, bool)
    keep[9] = False
    close(out[:, :4][..., keep], ref[:, :4][..., keep], v0[:1, :, keep], 4)
    close(out[:, 4:], ref[:, 4:], v0[1:], 4)
    k[1, 40, 2] = np.nan
    out = attend_f32(prompt_be, q, k, v0, n_head)
    assert np.all(np.isnan(out[40:, 4:])) and np.all(np.isfinite(out[:40, 4:])) and np.all(np.isfinite(out[:, :4]))


def attend_f32(b, q, k, v, n_head):
    n_kv, kv_len, hd = k.shape
    c = A.KVCache(b, kv_len, 1, n_kv, hd)
    c.append(0, k, v, kv_len, hd, mem=B.MEM_HOST)
    out = A.compute_attention(b, dev(q), c, 0, n_head, n_kv, hd, q.shape[1], kv_len, kv_len - q.shape[1]).cpu().numpy()
    c.close()
    return out


@pytest.mark.parametrize("n_head,n_kv,hd", [(32, 8, 128), (8, 8, 64), (24, 8, 128), (6, 4, 64)])
@pytest.mark.parametrize("q_len,start", [(2, 3000), (9, 1200), (40, 0), (64, 700), (230, 0)])
def test_the_rule_changes_no_result(be, prompt_be, n_head, n_kv, hd, q_len, start):
    """Whichever kernel the rule takes, the other agrees."""
    r = np.random.default_rng(q_len)
    kv_len = start + q_len
    q, k, v = (r.standard_normal(s).astype(F32) for s in ((n_head, q_len, hd), (n_kv, kv_len, hd), (n_kv, kv_len, hd)))
    rows = backend(1 << 30)
    outs = [attend_f32(b, q, k, v, n_head) for b in (be, prompt_be, rows)]
    rows.close()
    assert np.array_equal(outs[0], outs[1]) or np.array_equal(outs[0], outs[2])
    close(outs[1], outs[2], v, n_head)


# ---- weights and values far apart ------------------------------------------------

def exact(q, k, v, n_head):
    """In 64 bits; the queries are the last ones."""
    n_kv, kv_len, hd = k.shape
    q_len = q.shape[1]
    out = np.empty((q_len, n_head, hd))
    with np.errstate(over="ignore", invalid="ignore"):
        for h in range(n_head):
            j = h * n_kv // n_head
            s = q[h].astype(np.float64) @ k[j].astype(np.float64).T / np.sqrt(hd)
            s[np.arange(kv_len)[None, :] > kv_len - q_len + np.arange(q_len)[:, None]] = -np.inf
            p = np.exp(s - s.max(1, keepdims=True))
            out[:, h] = p @ v[j].astype(np.float64) / p.sum(1, keepdims=True)
    return out


def sink(r, n_head, n_kv, q_len, kv_len, hd, at, gap):
    """Every query scores position `at` `gap` nats above the largest other one."""
    a = np.zeros(hd)
    a[0] = 1.0
    q = r.standard_normal((n_head, q_len, hd)) * 0.1
    q[:, :, 0] = np.sqrt(hd)
    k = r.standard_normal((n_kv, kv_len, hd))
    k[:, at] = 0.0
    k[:, at, 0] = np.delete(k[:, :, 0], at, 1).max(1) + gap
    return q.astype(F32), k.astype(F32), r.standard_normal((n_kv, kv_len, hd)).astype(F32)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("kv_len,gap,top", [
    (1024, 12, 0.0), (1024, 16, 0.0), (4096, 20, 0.0), (4096, 20, 1.0), (200, 12, 1e-6), (33, 12, 0.0),
])
def test_small_weights_keep_their_bits(prompt_be, hd, kv_len, gap, top):
    """One position takes all but e^-gap of the weight and its V is `top` times
    as large as the others': with 0 the results are the small weights' own.
    Bar, relative to each head's results: a score of s nats rounds to s 2^-24,
    and so does its weight's exponent; 2^-22 s leaves room for the products'
    own roundings (s: the gap and 5 nats of the others' scores)."""
    n_head, n_kv, q_len = 8, 2, 32
    r = np.random.default_rng(kv_len + gap)
    q, k, v = sink(r, n_head, n_kv, q_len, kv_len, hd, 0, gap)
    v[:, 0] *= F32(top)
    out, ref = attend_f32(prompt_be, q, k, v, n_head), exact(q, k, v, n_head)
    for h in range(n_head):
        # the first query of 33 positions sees two of them: rows on their own
        err = np.linalg.norm(out[:, h] - ref[:, h], axis=1) / np.linalg.norm(ref[:, h], axis=1)
        assert np.max(err) <= (gap + 5) * 2.0 ** -22, (h, float(np.max(err)))


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("big", [1e4, 1e8, 1e10, 1e30, 3e38])
@pytest.mark.parametrize("where", ["masked", "weightless", "grown", "first"])
def test_values_beside_a_large_one(prompt_be, hd, big, where):
    """A large finite V that a row gives no weight costs the row nothing: at a
    later position of its block, at an earlier position whose weight is 0, or
    in blocks that it sees nothing of.  "first": at the position that takes all
    the weight, where the result is as large.  Bar 2e-6 of the largest |V| that
    the row gives weight to, per dim."""
    n_head, n_kv, q_len, kv_len = 8, 2, 90, 90
    r = np.random.default_rng(int(np.log10(big)))
    at = {"masked": 45, "weightless": 3, "grown": 70, "first": 0}[where]
    q, k, v = sink(r, n_head, n_kv, q_len, kv_len, hd, at, -400.0 if where == "weightless" else 30.0 if where == "first" else 0.0)
    v[:, at, 5:9] = F32(big)
    rows = np.arange(at) if where in ("masked", "grown") else np.arange(at + 1, q_len) if where == "weightless" else np.arange(q_len)
    out, ref = attend_f32(prompt_be, q, k, v, n_head), exact(q, k, v, n_head)
    seen = np.abs(v[:, :kv_len]).copy()
    if where != "first":
        seen[:, at] = 0.0
    for h in range(n_head):
        top = np.maximum.accumulate(seen[h * n_kv // n_head], axis=0)[rows]
        err = np.abs(out[rows, h] - ref[rows, h])
        assert np.all(err <= 2e-6 * top), (h, float(np.max(err / top)))


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("octaves", [20, 26, 29, 31, 32, 33.5, 35])
def test_values_of_one_size_beside_a_large_one(prompt_be, hd, octaves):
    """All |V| between 1 and 2 but for one masked position, 2^octaves: up to 31
    octaves the split holds them (to 2^-20 at worst), above that the f32
    products take the tile.  Bar 2^-20 of the largest |V| for a value and as
    much for the weights' own roundings (scores below 10 nats to 2^-22)."""
    n_head, n_kv, q_len, at = 8, 2, 64, 50
    r = np.random.default_rng(hd)
    q, k = (r.standard_normal(s).astype(F32) for s in ((n_head, q_len, hd), (n_kv, q_len, hd)))
    v = ((1 + r.random((n_kv, q_len, hd))) * r.choice([-1.0, 1.0], (n_kv, 1, hd))).astype(F32)
    v[:, at] = F32(2.0 ** octaves)
    out, ref = attend_f32(prompt_be, q, k, v, n_head), exact(q, k, v, n_head)
    assert np.max(np.abs(out[:at] - ref[:at])) <= 2 * 2.0 * 2.0 ** -20


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("case", ["1e6", "1e8", "1e30", "huge keys", "huge queries"])
def test_keys_and_queries_beside_large_elements(prompt_be, hd, case):
    """A large key element that the queries do not touch (they are 0 there)
    leaves the scores alone, and so do scales that only the product evens out.
    Bar 4e-6 of the largest |V|: scores of 10 nats to 2^-22."""
    n_head, n_kv, q_len, kv_len = 8, 2, 100, 160
    r = np.random.default_rng(hd)
    q, k, v = (r.standard_normal(s).astype(F32) for s in ((n_head, q_len, hd), (n_kv, kv_len, hd), (n_kv, kv_len, hd)))
    if case == "huge keys":        # one row in ten, against tiny queries: ordinary scores
        k[:, ::10] *= F32(1e33)
        q *= F32(1e-33)
    elif case == "huge queries":   # a query row in ten against keys that are all tiny
        q[:, ::10] *= F32(1e33)
        k *= F32(1e-33)
    else:
        q[:, :, 7] = 0.0
        k[:, 20:120:3, 7] = F32(float(case))
    out, ref = attend_f32(prompt_be, q, k, v, n_head), exact(q, k, v, n_head)
    for h in range(n_head):
        top = np.max(np.abs(v[h * n_kv // n_head]), axis=0)
        err = np.abs(out[:, h] - ref[:, h])
        assert np.all(err <= 4e-6 * top), (h, float(np.max(err / top)))


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("q_len,start,at", [(70, 0, 5), (70, 0, 40), (8, 300, 305), (100, 600, 640)])
def test_infinities_and_nan_that_only_later_rows_see(prompt_be, orc, hd, q_len, start, at):
    """Infinities and NaN in V and K at position `at` change no earlier row, also
    of its block of 32 positions, and no other dim or head; the last case runs
    in pieces."""
    n_head, n_kv, kv_len = 8, 2, start + q_len
    r = np.random.default_rng(q_len + at)
    q, k, v = (r.standard_normal(s).astype(F32) for s in ((n_head, q_len, hd), (n_kv, kv_len, hd), (n_kv, kv_len, hd)))
    ref = orc.attention(q, k, v, n_head, q_len, kv_len, start)
    bad = v.copy()
    bad[0, at, 9], bad[0, at, 10], bad[0, at, 11] = np.inf, -np.inf, np.nan
    out = attend_f32(prompt_be, q, k, bad, n_head)
    late = np.arange(q_len) >= at - start
    assert np.all(np.isposinf(out[late, :4, 9])) and np.all(np.isneginf(out[late, :4, 10])) and np.all(np.isnan(out[late, :4, 11]))
    out[late, :4, 9:12] = ref[late, :4, 9:12]
    close(out, ref, v, n_head)
    bad = k.copy()
    bad[1, at, 3] = np.nan
    out = attend_f32(prompt_be, q, bad, v, n_head)
    assert np.all(np.isnan(out[late, 4:]))
    out[late, 4:] = ref[late, 4:]
    close(out, ref, v, n_head)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("n_head,n_kv,q_len,start", [(14, 2, 8, 700), (15, 5, 40, 300), (71, 1, 5, 400), (3, 1, 70, 200), (1, 1, 33, 100)])
@pytest.mark.parametrize("pieces", [0, 3])
def test_heads_of_no_whole_q8_k_blocks(orc, monkeypatch, hd, n_head, n_kv, q_len, start, pieces):
    """Heads times dims that are no multiple of 256 in pieces too: the last wave
    of the merge has rows of fewer heads."""
    if pieces:
        monkeypatch.setenv("BARQ_ATTN_MFMA_SPLIT", str(pieces))
    b = backend(1)
    r = np.random.default_rng(n_head)
    kv_len = start + q_len
    q, k, v = (r.standard_normal(s).astype(F32) for s in ((n_head, q_len, hd), (n_kv, kv_len, hd), (n_kv, kv_len, hd)))
    out = attend_f32(b, q, k, v, n_head)
    b.close()
    close(out, orc.attention(q, k, v, n_head, q_len, kv_len, start), v, n_head)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("pieces", [0, 2])
def test_outputs_at_any_float(orc, monkeypatch, hd, pieces):
    """The output need only be 4-byte aligned; what stands around it stays."""
    import torch
    if pieces:
        monkeypatch.setenv("BARQ_ATTN_MFMA_SPLIT", str(pieces))
    b = backend(1)
    n_head, n_kv, q_len, kv_len = 6, 2, 50, 100
    r = np.random.default_rng(hd)
    q, k, v = (r.standard_normal(s).astype(F32) for s in ((n_head, q_len, hd), (n_kv, kv_len, hd), (n_kv, kv_len, hd)))
    c = A.KVCache(b, kv_len, 1, n_kv, hd)
    c.append(0, k, v, kv_len, hd, mem=B.MEM_HOST)
    n = q_len * n_head * hd
    buf, qd = torch.full((n + 8,), 7.0, device="cuda"), dev(q)
    torch.cuda.synchronize()
    for at in (1, 2, 3):
        buf.fill_(7.0)
        torch.cuda.synchronize()
        B._lib.check(b._lib.barq_rocm_attention(b.h, qd.data_ptr(), c.c, 0, n_head, n_kv, hd, q_len, kv_len, kv_len - q_len,
                                                buf.data_ptr() + 4 * at, B.MEM_DEVICE))
        b.sync()
        got = buf.cpu().numpy()
        assert np.all(got[:at] == 7.0) and np.all(got[at + n:] == 7.0)
        close(got[at:at + n].reshape(q_len, n_head, hd), orc.attention(q, k, v, n_head, q_len, kv_len, kv_len - q_len), v, n_head)
    c.close()
    b.close()
