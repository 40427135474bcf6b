"""The form a decode call takes by its shape (query heads per wave, waves, one launch or split).

Batches at the edges of each choice (128 to 3072 workgroups, 256 to 1024 keys) against the oracle, and
the calls that must stay on the one-launch kernel because they bring no workspace.
"""

import numpy as np
import pytest
import torch

import oracle.attention as oa
from femtovllm import workloads
from helpers import assert_close, np32, np64, np_tables

pytestmark = pytest.mark.gpu

# (heads, kv_heads, sequences): on both sides of the workgroup counts where the form changes
SHAPES = [(16, 8, 16), (16, 8, 17), (16, 8, 32), (16, 8, 33), (32, 8, 32), (32, 8, 33), (64, 8, 8), (64, 8, 17),
          (64, 8, 33), (64, 8, 65), (64, 8, 193), (16, 8, 8), (16, 8, 193), (4, 1, 65), (3, 3, 86), (24, 2, 11)]


def _batch(heads, kv_heads, seqs, longest, dtype):
    lens = [int(x) for x in np.random.default_rng(seqs).integers(1, 40, size=seqs)]
    lens[seqs // 2] = longest
    w = workloads.make_paged_workload("route", [(n - 1, 1) for n in lens], heads, kv_heads, seed=seqs, dtype=dtype)
    return w


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("longest", [200, 300, 513, 900, 1025])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_route_edges(ops, gpu, dtype, longest, shape):
    w = _batch(*shape, longest, dtype)
    q, meta = w.gemv_call(device=gpu)
    wd = w.to(gpu)
    out = ops.paged_attention_gemv(q.to(gpu), wd.k_pool, wd.v_pool, meta.block_tables, meta.kv_lens, meta.max_kv_len)
    torch.cuda.synchronize()
    want = oa.paged_decode(np64(q), np32(w.k_pool), np32(w.v_pool), np_tables(meta), meta.kv_lens.tolist())
    assert_close(out, want, dtype, f"decode route {shape} {longest} {dtype}")


# (heads, kv_heads, sequences, longest): on both sides of the lines by key count, rounds and head ratio
LINES = [(8, 1, 137, 128), (8, 1, 137, 129), (64, 8, 34, 512), (64, 8, 34, 513), (64, 8, 65, 257), (24, 2, 21, 768),
         (24, 2, 21, 769), (16, 8, 24, 500), (16, 8, 25, 500), (2, 1, 256, 1000)]


@pytest.mark.parametrize("shape", LINES, ids=str)
def test_route_lines(ops, gpu, shape):
    w = _batch(*shape, torch.bfloat16)
    q, meta = w.gemv_call(device=gpu)
    wd = w.to(gpu)
    out = ops.paged_attention_gemv(q.to(gpu), wd.k_pool, wd.v_pool, meta.block_tables, meta.kv_lens, meta.max_kv_len)
    want = oa.paged_decode(np64(q), np32(w.k_pool), np32(w.v_pool), np_tables(meta), meta.kv_lens.tolist())
    assert_close(out, want, torch.bfloat16, f"decode route {shape}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_no_workspace_within_the_limit(gpu, dtype):
    """A shape that would run split, called with no workspace: one launch, as before."""
    from femtovllm import _C

    w = _batch(64, 8, 193, 1000, dtype)
    q, meta = w.gemv_call(device=gpu)
    wd, q = w.to(gpu), q.to(gpu).contiguous()
    out = torch.empty_like(q)
    k, v, t = wd.k_pool, wd.v_pool, meta.block_tables
    rc = _C._lib.femto_paged_attention_gemv(
        _C._DTYPE[dtype], q.data_ptr(), q.stride(0), q.stride(1), out.data_ptr(), out.stride(0), out.stride(1), k.data_ptr(),
        v.data_ptr(), *k.shape, *k.stride()[:3], t.data_ptr(), t.size(1), t.stride(0), meta.kv_lens.data_ptr(), q.size(1),
        q.size(0), meta.max_kv_len, None, 0, _C._stream(q.device))
    assert rc == 0, _C._lib.femto_attn_last_error().decode()
    torch.cuda.synchronize()
    want = oa.paged_decode(np64(q), np32(w.k_pool), np32(w.v_pool), np_tables(meta), meta.kv_lens.tolist())
    assert_close(out, want, dtype, "no workspace")


@pytest.mark.parametrize("heads", [(16, 8), (16, 16)], ids=str)
@pytest.mark.parametrize("keys", [1030, 1500, 2900])
def test_infinite_values_stay_infinite(ops, gpu, heads, keys):
    """Equal scores, and V infinite in the first key and in the last page of one dim each: both merges of split
    contexts (the merge launch, and the one in a prefill call's launch) give infinities there and the mean of
    V elsewhere, whatever the number of slots."""
    w = workloads.make_paged_workload("inf", [(keys - 1, 1), (20, 9)], *heads, seed=61, poison=False)
    q, meta = w.gemm_call(device=gpu)
    wd = w.to(gpu)
    wd.k_pool.zero_()
    table = meta.block_tables[0].tolist()
    wd.v_pool[table[0], :, 0, 3] = float("inf")
    wd.v_pool[table[(keys - 1) // 16], :, 0, 5] = float("-inf")
    q = q.to(gpu)
    v = wd.v_pool[torch.tensor(table[: (keys + 15) // 16], device=gpu)].float().permute(1, 0, 2, 3).flatten(1, 2)[:, :keys]
    want = v.mean(1).repeat_interleave(heads[0] // heads[1], 0)
    rows = [ops.paged_attention_gemv(q[:, :1], wd.k_pool, wd.v_pool, meta.block_tables[:1], meta.kv_lens[:1], keys)[:, 0],
            ops.paged_attention_gemm(q, wd.k_pool, wd.v_pool, meta.cu_seqlens, meta.max_q_len, meta.Q_TILE_SIZE,
                                     meta.cu_q_tiles, meta.q_tile_to_seq_idx, meta.block_tables, meta.kv_lens,
                                     meta.positions)[:, 0]]
    for got in rows:
        assert torch.isposinf(got[:, 3]).all() and torch.isneginf(got[:, 5]).all()
        rest = [d for d in range(128) if d not in (3, 5)]
        # probabilities 1/n rounded to bf16 cancel in the quotient; the output rounding is 2^-9 relative
        assert torch.allclose(got[:, rest].float(), want[:, rest], rtol=2.0 ** -8, atol=1e-4)


@pytest.mark.parametrize("shape", [((64, 8), 100), ((16, 8), 8), ((32, 8), 200)], ids=str)
def test_captured_call_within_the_limit_holds_no_workspace(ops, gpu, shape):
    """f32 shapes that run split within 1024 keys: captured in a graph they are one launch (the routes sum in
    different orders, so equal bits tell which one ran), and replays still match after the stream's workspace
    was replaced by a larger one and its memory taken by another tensor."""
    from femtovllm import _C

    (heads, kv_heads), seqs = shape
    lens = [int(x) for x in np.random.default_rng(seqs).integers(600, 1000, size=seqs)]
    lens[0] = 1000
    w = workloads.make_paged_workload("capture", [(n - 1, 1) for n in lens], heads, kv_heads, seed=seqs,
                                      dtype=torch.float32)
    q, meta = w.gemv_call(device=gpu)
    wd, q = w.to(gpu), q.to(gpu).contiguous()
    call = lambda: ops.paged_attention_gemv(q, wd.k_pool, wd.v_pool, meta.block_tables, meta.kv_lens, meta.max_kv_len)

    def forced(limit):
        prev = _C._lib.femto_attn_set_decode_single_max_kv(limit)
        try:
            return call()
        finally:
            _C._lib.femto_attn_set_decode_single_max_kv(prev)

    one, split = forced(1 << 30), forced(-1)
    assert not torch.equal(one, split) and torch.equal(call(), split)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()  # this stream's workspace
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            out = call()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, one)
    old = _C._workspaces[(gpu.index, side.cuda_stream)]
    size = old.numel()
    with torch.cuda.stream(side):
        _C._decode_workspace(gpu, 2 * seqs, heads, 8192)
        del old
        other = torch.full((size,), 77, dtype=torch.uint8, device=gpu)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, one) and bool((other == 77).all())
