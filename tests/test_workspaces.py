"""Workspaces of the Python layer: what happens to one that a larger call replaces.

A graph captured while a workspace was in use writes its memory at every
replay, so the memory stays allocated when a later call on the stream needs
more.
"""

import weakref

import numpy as np
import pytest
import torch

import oracle.attention as oa
from femtovllm import workloads
from helpers import assert_close, np32, np64, np_tables


def test_replaced_workspaces_stay_allocated_and_bounded(monkeypatch):
    from femtovllm import _C

    monkeypatch.setattr(_C, "_stream", lambda device: 0)
    monkeypatch.setattr(_C, "_replaced_workspaces", [], raising=False)
    cache, seen = {}, []
    device = torch.device("cpu")
    for nbytes in (1000, 900, 1001, 1 << 16, (1 << 16) + 1, 1 << 20):
        ptr, size = _C._cached_workspace(cache, device, nbytes, zero=True)
        assert ptr % 256 == 0 and size >= nbytes
        (ws,) = cache.values()
        assert not ws.any() and ws.data_ptr() <= ptr < ws.data_ptr() + 256
        if not seen or seen[-1]() is not ws:
            seen.append(weakref.ref(ws))
        del ws
    assert len(seen) > 2
    assert all(r() is not None for r in seen), "a replaced workspace was freed"
    assert sum(r().numel() for r in seen[:-1]) < seen[-1]().numel()


@pytest.mark.parametrize("name,function", [("gemv", "_decode_workspace"), ("gemm", "_prefill_workspace")])
def test_a_replaced_workspace_function_is_asked(monkeypatch, name, function):
    """The native call looks the stream's workspace up by itself, so it is left out once the function is not
    the module's own."""
    from femtovllm import _C

    asked = []

    class Native:
        def __getattr__(self, entry):
            return lambda *args: asked.append(entry)

    q, pool, i32 = torch.zeros(2, 1, 128), torch.zeros(1, 1, 16, 128), torch.zeros(1, dtype=torch.int32)
    call = {"gemv": lambda: _C.PagedAttentionGemvCuda(q, pool, pool, i32[None], i32, 1),
            "gemm": lambda: _C.PagedAttentionGemmCuda(q, pool, pool, i32, 1, i32[None], i32, i32)}[name]
    monkeypatch.setattr(_C, "_native", Native())
    with pytest.raises(RuntimeError, match="GPU tensor"):
        call()
    assert asked == [name]
    monkeypatch.setattr(_C, function, lambda *args: (None, 0))
    with pytest.raises(RuntimeError, match="GPU tensor"):
        call()
    assert asked == [name]


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["decode", "prefill"])
def test_replay_after_the_workspace_grew(ops, gpu, entry):
    """Split decode (2000 keys) and a prefill call with split keys and decode rows, captured; then a larger
    call on the stream replaces the workspace and other tensors are allocated: replays stay right and leave
    those tensors alone."""
    from femtovllm import _C

    chunks = [(1999, 1), (300, 1), (6000, 40), (20, 70)] if entry == "prefill" else [(1999, 1), (300, 1), (1200, 1)]
    w = workloads.make_paged_workload("grow", chunks, 16, 8, seed=5)
    q, meta = w.gemm_call(device=gpu)
    wd, qd = w.to(gpu), q.to(gpu).contiguous()
    if entry == "prefill":
        call = lambda: ops.paged_attention_gemm(qd, wd.k_pool, wd.v_pool, meta.cu_seqlens, meta.max_q_len,
                                                meta.Q_TILE_SIZE, meta.cu_q_tiles, meta.q_tile_to_seq_idx,
                                                meta.block_tables, meta.kv_lens, meta.positions)
        want = oa.paged_prefill(np64(q), np32(w.k_pool), np32(w.v_pool), meta.raw_cu_seqlens, np_tables(meta),
                                meta.kv_lens.tolist(), np.array(meta.raw_positions))
        cache, grow = _C._prefill_workspaces, lambda: _C._prefill_workspace(gpu, 64, 128, 65, 16, 8, 4096)
    else:
        call = lambda: ops.paged_attention_gemv(qd, wd.k_pool, wd.v_pool, meta.block_tables, meta.kv_lens, 2000)
        want = oa.paged_decode(np64(q), np32(w.k_pool), np32(w.v_pool), np_tables(meta), meta.kv_lens.tolist())
        cache, grow = _C._workspaces, lambda: _C._decode_workspace(gpu, 64, 16, 8192)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()  # this stream's workspace
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            out = call()
        key = (gpu.index, side.cuda_stream)
        size = cache[key].numel()
        grow()
        assert cache[key].numel() >= 2 * size
        others = [torch.full((size,), 77, dtype=torch.uint8, device=gpu) for _ in range(3)]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_close(out, want, torch.bfloat16, f"{entry}, replay after the workspace grew")
        assert all(bool((x == 77).all()) for x in others)
