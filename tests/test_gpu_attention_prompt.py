"""The prompt attention kernel (split-f16 matrix products) on its own: tile
and block edges, value ranges its scales have to follow, values that are not
finite, and the rule that chooses it.  Parity against the oracle
(models/src/transformer.rs:301-374).

Bar: 2e-5 of the largest |V| of the same output dim.  Outputs are convex
combinations of V rows, and a score is a dot product of 64 or 128 terms, each
to 2^-24 of |q||k|, so at the sizes here (|score| below 10) a weight is off by
less than 10 * 2^-22 and an output by less than 1e-5 of the largest |V|.
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
    the positions, one dim zero for two blocks, one zero throughout)."""
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
    # a row's results only depend on what it sees: the bar per row uses V up to it
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
