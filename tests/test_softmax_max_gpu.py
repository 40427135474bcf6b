"""The running maximum of the tile kernel's softmax.

The kernel takes a block's exponentials against the running max it has, and
moves that max where a row's sum grew by more than 2^8.  The weights are
rounded to the storage type (the reference's Triton kernel does too,
femtovllm/ops/triton/paged_attention/paged_attention_gemm.py:153-155), so
which maximum they are relative to shows in the last bit of the outputs.
"""

import numpy as np
import pytest
import torch

from helpers import np64

pytestmark = pytest.mark.gpu

LOG2E = 1.4426950408889634


def rand(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g, dtype=torch.float32).to(dtype)


def round_to(x: np.ndarray, dtype) -> np.ndarray:
    return np64(torch.from_numpy(x).to(torch.float32).to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("entry,keys", [("dense", 33), ("dense", 50), ("dense", 64), ("paged", 64)])
def test_weights_of_the_first_tile_are_relative_to_its_maximum(ops, gpu, dtype, entry, keys):
    """Rows of up to 64 keys whose largest score lies in the second 32: the largest weight is 1 exactly,
    so outputs are the 64-bit result of weights rounded relative to the maximum over all keys, rounded once
    more.  Equal but for f32 rounding at a tie: of the output (2^-23 x 64 keys against 2^-9: < 1 %) or of a
    weight (of 64, each within f32 rounding of a tie with probability ~2^-12; such a weight moves a fifth of
    the row's outputs at most: < 1 %).  With a maximum over the first 32 keys only, 45 % of those outputs
    differ (64 keys, f16)."""
    from femtovllm import _C

    H, T = 2, 64
    q = rand((H, T, 128), dtype, 1)
    k = rand((H, keys, 128), dtype, 2)
    v = rand((H, keys, 128), dtype, 3)
    k[:, 32:] *= 1.5
    if entry == "dense":
        out = _C.FlashAttentionWarpCuda(q[None].to(gpu), k[None].to(gpu), v[None].to(gpu))[0]
        see = np.full(T, keys)
    else:
        pool = lambda x: x.reshape(H, keys // 16, 16, 128).transpose(0, 1).contiguous().to(gpu)
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=gpu)
        out = ops.paged_attention_gemm(q.to(gpu), pool(k), pool(v), i32([0, T]), T, 32, i32([0, 2]), i32([0, 0]),
                                       i32([list(range(keys // 16))]), i32([keys]), i32(list(range(T))))
        see = np.arange(1, T + 1)
    s = np64(q) @ np64(k).transpose(0, 2, 1) * (LOG2E / np.sqrt(128.0))
    s = np.where(np.arange(keys)[None, None, :] < see[None, :, None], s, -np.inf)
    in_second = s.argmax(-1) >= 32
    assert in_second.mean() > (0.1 if keys == 33 else 0.3)
    p = round_to(np.exp2(s - s.max(-1, keepdims=True)), dtype)
    want = round_to(p @ np64(v) / p.sum(-1, keepdims=True), dtype)
    same = np64(out) == want
    assert same[in_second].mean() > 0.97, f"{(1 - same[in_second].mean()) * 100:.1f} % differ"
    assert same.mean() > 0.97


def _paged(monkeypatch, ops, gpu, chunks, heads, dtype, dim, change, split):
    """A prefill call over pools that ``change(k, rows)`` altered (``k`` the float K pool, ``rows(s, j)`` the
    index of key j of sequence s in it) and its oracle result."""
    import oracle.attention as oa
    from femtovllm import _C, workloads
    from helpers import np32, np_tables

    w = workloads.make_paged_workload("softmax", chunks, *heads, seed=3, dtype=dtype, head_dim=dim)
    q, meta = w.gemm_call(device=gpu)
    tables = meta.block_tables.tolist()
    k = w.k_pool.float()
    change(q, k, lambda s, j: (tables[s][j // 16], slice(None), j % 16))
    w.k_pool.copy_(k.to(dtype))
    wd = w.to(gpu)
    with monkeypatch.context() as m:
        if not split:
            m.setattr(_C, "_prefill_workspace", lambda *args: (None, 0))
        out = ops.paged_attention_gemm(q.to(gpu), wd.k_pool, wd.v_pool, meta.cu_seqlens, meta.max_q_len, meta.Q_TILE_SIZE,
                                       meta.cu_q_tiles, meta.q_tile_to_seq_idx, meta.block_tables, meta.kv_lens,
                                       meta.positions)
    with np.errstate(invalid="ignore"):
        want = oa.paged_prefill(np64(q), np32(w.k_pool), np32(w.v_pool), meta.raw_cu_seqlens, np_tables(meta),
                                meta.kv_lens.tolist(), np.asarray(meta.raw_positions))
    return out, want


@pytest.mark.parametrize("dtype,heads,dim", [(torch.float16, (4, 2), 128), (torch.bfloat16, (4, 2), 128),
                                             (torch.bfloat16, (8, 2), 48)], ids=str)
@pytest.mark.parametrize("jump", [9.0, 60.0])
@pytest.mark.parametrize("at", [96, 127, 128, 159, 160, 168])
@pytest.mark.parametrize("beside", [False, True], ids=["alone", "beside_decode_rows"])
def test_scores_that_jump_at_the_causal_limit(ops, gpu, monkeypatch, dtype, heads, dim, jump, at, beside):
    """70 tokens after 99 cached keys, so the last tile is partly filled and all tiles from key 99 on are
    masked; scores of some rows jump (log2 units, times 1, -1 or 0 by row) at the first or last key of either
    32-key block, in rows that see the jump beside rows that do not."""
    from helpers import assert_close

    chunks = [(99, 70)] + ([(299, 1), (40, 1), (700, 1)] if beside else [(30, 2)])

    def change(q, k, rows):
        q[:, :70, 0] = torch.tensor([16.0, -16.0, 0.0]).repeat(24)[:70].to(q.dtype)
        for j in range(169):
            k[rows(0, j)][..., 0] = jump * np.sqrt(dim) / LOG2E / 16.0 if j >= at else 0.0

    out, want = _paged(monkeypatch, ops, gpu, chunks, heads, dtype, dim, change, split=beside)
    assert_close(out, want, dtype, f"jump {jump} at key {at} {heads} {dim} beside={beside}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rising", [True, False])
def test_pieces_whose_maxima_differ(ops, gpu, monkeypatch, dtype, rising):
    """A sequence cut into key pieces, its scores rising or falling by 12 log2 units every 500 keys: each
    piece's running max is far from the others', and the merge weighs them."""
    from helpers import assert_close

    def change(q, k, rows):
        q[:, :40, 0] = torch.tensor([16.0, -16.0, 0.0, 4.0]).repeat(10).to(q.dtype)
        for j in range(6040):
            step = j // 500 if rising else 12 - j // 500
            k[rows(0, j)][..., 0] = 12.0 * step * np.sqrt(128.0) / LOG2E / 16.0

    out, want = _paged(monkeypatch, ops, gpu, [(6000, 40), (20, 64)], (16, 8), dtype, 128, change, split=True)
    assert_close(out, want, dtype, f"pieces, rising={rising}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("at", [5, 40, 100, 140])
def test_infinite_and_nan_scores(ops, gpu, monkeypatch, dtype, value, at):
    """One key with an infinite or NaN element: rows whose score there is +inf or NaN are NaN, rows with -inf
    leave the key out, rows that do not see it are untouched."""
    from helpers import assert_close

    def change(q, k, rows):
        q[:, :70, 0] = torch.tensor([2.0, -2.0]).repeat(35).to(q.dtype)
        k[rows(0, at)][..., 0] = value

    out, want = _paged(monkeypatch, ops, gpu, [(99, 70), (30, 2)], (4, 2), dtype, 128, change, split=False)
    assert np.isnan(want).any() and not np.isnan(want).all()
    assert_close(out, want, dtype, f"{value} at key {at}")
