"""Tile choices of the batched GEMMs that depend on how many tiles a shape has."""
import os

import numpy as np
import pytest

import barq_rocm as B
from barq_rocm import synth

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def backend(**env):
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        return B.Backend(0)
    finally:
        for k, v in old.items():
            os.environ.pop(k) if v is None else os.environ.__setitem__(k, v)


@pytest.mark.parametrize("rows", [31, 32, 33, 41, 63, 64, 65, 129])
def test_expert_groups_of_64_row_tiles(be, rows):
    """Expert groups of 32 rows or more take 64-row tiles; a weight row's products
    are summed in the same order as on 32-row tiles, so the outputs are the
    same bits.  Three experts with `rows` - 20, `rows` and `rows` + 20 rows."""
    hidden, n_ff, ne = 512, 768, 3
    g, u = ([dev(synth.gen_q4_k(n_ff, hidden, 10 * e + s)) for e in range(ne)] for s in (1, 2))
    d = [dev(synth.gen_q6_k(hidden, n_ff, 10 * e + 3)) for e in range(ne)]
    ids = np.concatenate([np.full(rows + 20 * (e - 1), e) for e in range(ne)]).astype(np.int32)
    ids = np.random.default_rng(rows).permutation(ids)[:, None]
    x, w = synth.gen_f32(len(ids) * hidden, 5).reshape(-1, hidden), np.ones((len(ids), 1), np.float32)
    small = backend(BARQ_GEMM_BM="32")
    outs = [b.moe_ffn(B.Q4_K, g, B.Q4_K, u, B.Q6_K, d, hidden, n_ff, dev(x), len(ids), dev(ids), dev(w), 1,
                      B.ACT_F32_Q8).cpu().numpy() for b in (be, small)]
    small.close()
    assert np.any(outs[0]) and np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("t", [B.Q4_0, B.Q8_0, B.Q4_0_BARQ])
@pytest.mark.parametrize("n,m,scale", [
    (16400, 65, 1.0),     # 258 tiles of 64 rows: 32-row tiles, one K-group
    (17000, 192, 1.0),    # 399 tiles of 64 rows, more than three of 32 rows per CU: 64-row tiles, one K-group
    (21800, 130, 1.0),    # 513 tiles: 64-row tiles, one K-group
    (32800, 4, 1.0),      # more tiles than CUs for a few rows: 32-row tiles, one K-group
    (32800, 32, 1.0),
    (200, 70, 1e-6),      # activation scales that are subnormal in f16
    (200, 33, 3e4),       # large ones
])
def test_32_element_blocks_many_tiles(be, orc, t, n, m, scale):
    """Against the oracle at 1e-6: integer products are exact, the f16 scales'
    products too, and k / 32 = 8 terms are summed in f32."""
    k = 256
    w, x = synth.gen_weights(t, n, k, 7), synth.gen_f32(m * k, 8).reshape(m, k) * np.float32(scale)
    xq = be.quantize_act(B.Q8_0, dev(x))
    y = be.matmul(t, dev(w), n, k, B.Q8_0, xq, m).cpu().numpy()
    ref = orc.matmul(t, w, n, k, orc.Q8_0, xq.cpu().numpy(), m).reshape(m, n)
    err = np.linalg.norm(y.astype(np.float64) - ref) / np.linalg.norm(ref.astype(np.float64))
    assert np.any(ref) and err <= 1e-6, err


@pytest.mark.parametrize("n,k,m", [
    (16500, 256, 65),      # 258 tiles of 64 rows, 129 of 128: one round instead of two; ragged in both
    (16512, 768, 128),     # whole tiles, an odd number of super-blocks
    (11000, 512, 193),     # a last tile with one row in its upper half
    (16500, 512, 129),     # 258 tiles of 128 rows too: 64-row tiles stay
])
def test_q4_k_prompts_on_128_row_tiles(be, orc, n, k, m):
    """Against the oracle at 1e-6: a super-block's integer sums are exact and
    up to three of them are added in f32."""
    w, x = synth.gen_q4_k(n, k, 3), synth.gen_f32(m * k, 4).reshape(m, k)
    xq = be.quantize_act(B.Q8_K, dev(x))
    y = be.matmul(B.Q4_K, dev(w), n, k, B.Q8_K, xq, m).cpu().numpy()
    ref = orc.matmul(B.Q4_K, w, n, k, orc.Q8_K, xq.cpu().numpy(), m).reshape(m, n)
    err = np.linalg.norm(y.astype(np.float64) - ref) / np.linalg.norm(ref.astype(np.float64))
    assert np.any(ref) and err <= 1e-6, err


def test_expert_gather_of_more_blocks_than_workgroups(be):
    """1031 assignments of 8 blocks (some experts out of range): each wave
    quantizes several blocks, with the outputs of the two-launch form."""
    hidden, n_ff, ne, n = 2048, 512, 3, 1031
    g, u = ([dev(synth.gen_q4_k(n_ff, hidden, 10 * e + s)) for e in range(ne)] for s in (1, 2))
    d = [dev(synth.gen_q6_k(hidden, n_ff, 10 * e + 3)) for e in range(ne)]
    ids = np.random.default_rng(2).integers(-1, ne + 1, (n, 1)).astype(np.int32)
    x, w = synth.gen_f32(n * hidden, 5).reshape(n, hidden), np.ones((n, 1), np.float32)
    two = backend(BARQ_MOE_FUSED_GROUP="0")
    outs = [b.moe_ffn(B.Q4_K, g, B.Q4_K, u, B.Q6_K, d, hidden, n_ff, dev(x), n, dev(ids), dev(w), 1,
                      B.ACT_F32_Q8).cpu().numpy() for b in (be, two)]
    two.close()
    assert np.any(outs[0]) and np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("n,k,m", [(16500, 512, 65), (16512, 4096, 128), (11000, 1024, 193)])
def test_q4_k_128_row_tiles_sum_like_64_row_ones(be, n, k, m):
    """Two chains of f32 sums (even and odd super-blocks) on both: the same bits."""
    w, x = synth.gen_q4_k(n, k, 3), synth.gen_f32(m * k, 4).reshape(m, k)
    xq = be.quantize_act(B.Q8_K, dev(x))
    small = backend(BARQ_GEMM_BM="64")
    outs = [b.matmul(B.Q4_K, dev(w), n, k, B.Q8_K, xq, m).cpu().numpy() for b in (be, small)]
    small.close()
    assert np.any(outs[0]) and np.array_equal(outs[0], outs[1])


def test_q6_k_128_row_tiles_sum_like_64_row_ones(be):
    """One chain of f32 sums on both (no K slices at this width): the same bits."""
    n, k, m = 16512, 1024, 256
    w, x = synth.gen_q6_k(n, k, 3), synth.gen_f32(m * k, 4).reshape(m, k)
    xq = be.quantize_act(B.Q8_K, dev(x))
    small = backend(BARQ_GEMM_BM="66")
    outs = [b.matmul(B.Q6_K, dev(w), n, k, B.Q8_K, xq, m).cpu().numpy() for b in (be, small)]
    small.close()
    assert np.any(outs[0]) and np.array_equal(outs[0], outs[1])
