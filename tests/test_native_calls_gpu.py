"""The calls' native path (femto_native) against the Python path behind it.

Both run the same kernels, so over the forms that the calls accept (strides, types, given outputs) the
results are the same bytes, and what the Python path refuses is refused with its own message.
"""

import pytest
import torch

from femtovllm import workloads

pytestmark = pytest.mark.gpu


class _NoNative:
    def __getattr__(self, name):
        return lambda *args: None


class _Recorder:
    """The native module, noting which entry took a call (returned a tensor) and which declined."""

    def __init__(self, native):
        self.native, self.took, self.declined = native, [], []

    def __getattr__(self, name):
        def call(*args):
            out = getattr(self.native, name)(*args)
            (self.declined if out is None else self.took).append(name)
            return out

        return call


def _both(monkeypatch, call, entry):
    """The Python path first (it makes the stream's workspace), then the native one, which has to take the call."""
    from femtovllm import _C

    with monkeypatch.context() as m:
        m.setattr(_C, "_native", _NoNative())
        want = call()
    recorder = _Recorder(_C._native)
    with monkeypatch.context() as m:
        m.setattr(_C, "_native", recorder)
        got = call()
    torch.cuda.synchronize()
    assert recorder.took == [entry] and not recorder.declined
    assert got.shape == want.shape and got.stride() == want.stride() and got.dtype == want.dtype
    assert torch.equal(got.nan_to_num(nan=7.0), want.nan_to_num(nan=7.0))
    return got


def _forms(q):
    """q (heads, tokens, dim) as the engine passes it, contiguous, and as part of a wider tensor."""
    wide = torch.zeros(q.size(1), q.size(0) + 3, q.size(2), dtype=q.dtype, device=q.device)
    wide[:, 1:-2] = q.transpose(0, 1)
    return {"transposed": q.transpose(0, 1).contiguous().transpose(0, 1), "contiguous": q.contiguous(),
            "slice": wide[:, 1:-2].transpose(0, 1)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [128, 64])
@pytest.mark.parametrize("lens", [[17, 300, 1], [5, 1500]], ids=str)
def test_decode(ops, gpu, monkeypatch, dtype, dim, lens):
    w = workloads.make_paged_workload("native_decode", [(n - 1, 1) for n in lens], 4, 2, seed=51, dtype=dtype, head_dim=dim)
    q, meta = w.gemv_call(device=gpu)
    wd = w.to(gpu)
    for form, qf in _forms(q.to(gpu)).items():
        tables = meta.block_tables
        if form == "slice":  # a table with a wider row stride
            wide = torch.full((tables.size(0), tables.size(1) + 5), -1, dtype=torch.int32, device=gpu)
            wide[:, : tables.size(1)] = tables
            tables = wide[:, : tables.size(1)]
        _both(monkeypatch, lambda: ops.paged_attention_gemv(qf, wd.k_pool, wd.v_pool, tables, meta.kv_lens, meta.max_kv_len), "gemv")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [128, 48])
def test_prefill(ops, gpu, monkeypatch, dtype, dim):
    w = workloads.make_paged_workload("native_prefill", [(40, 33), (700, 1), (0, 5)], 4, 2, seed=52, dtype=dtype, head_dim=dim)
    q, meta = w.gemm_call(device=gpu)
    wd = w.to(gpu)
    for qf in _forms(q.to(gpu)).values():
        _both(monkeypatch, lambda: ops.paged_attention_gemm(
            qf, wd.k_pool, wd.v_pool, meta.cu_seqlens, meta.max_q_len, meta.Q_TILE_SIZE, meta.cu_q_tiles,
            meta.q_tile_to_seq_idx, meta.block_tables, meta.kv_lens, meta.positions), "gemm")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("given", [False, True])
def test_prologue(ops, gpu, monkeypatch, dtype, packed, given):
    from femtovllm.rope import rope_tables

    w = workloads.make_paged_workload("native_prologue", [(40, 33), (700, 1), (0, 5)], 4, 2, seed=53, dtype=dtype, poison=False)
    _, meta = w.gemm_call(device=gpu)
    wd = w.to(gpu)
    n = sum(x for _, x in [(40, 33), (700, 1), (0, 5)])
    qkv = torch.randn(n, 8, 128, generator=torch.Generator().manual_seed(1)).to(dtype).to(gpu)
    q, k, v = (x if packed else x.contiguous() for x in qkv.split([4, 2, 2], dim=1))
    weight = torch.linspace(0.5, 1.5, 128, device=gpu).to(dtype)
    cos, sin = rope_tables(1024, 128, device=gpu)

    def call():
        kp, vp = wd.k_pool.clone(), wd.v_pool.clone()
        out = torch.empty(n, 6, 128, dtype=dtype, device=gpu)[:, 1:5] if given else None
        r = ops.qk_norm_rope_cache_write(q, k, v, weight, weight, 1e-6, cos, sin, meta.positions, kp, vp, meta.block_tables,
                                         cu_seqlens=meta.cu_seqlens, max_q_len=meta.max_q_len, out=out)
        assert out is None or r is out
        return torch.cat([r.reshape(-1), kp.reshape(-1), vp.reshape(-1)])

    _both(monkeypatch, call, "prologue")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 4, 2, 70, 200), (2, 8, 8, 1, 33), (3, 6, 2, 129, 1)], ids=str)
def test_dense(gpu, monkeypatch, dtype, shape):
    from femtovllm import _C

    B, H, KVH, Tq, Tk = shape
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(s, generator=g).to(dtype).to(gpu) for s in ((B, H, Tq, 128), (B, KVH, Tk, 128), (B, KVH, Tk, 128)))
    _both(monkeypatch, lambda: _C.FlashAttentionWarpCuda(q, k, v), "flash")


def test_forms_left_to_the_python_path(ops, gpu, monkeypatch):
    """A first call on a stream (no workspace yet), a subclass and a float max_kv_len: declined, the same result."""
    from femtovllm import _C

    class Sub(torch.Tensor):
        pass

    w = workloads.make_paged_workload("declined", [(1499, 1), (20, 1)], 4, 2, seed=55)
    q, meta = w.gemv_call(device=gpu)
    wd, q = w.to(gpu), q.to(gpu)
    call = lambda q=q, n=meta.max_kv_len: ops.paged_attention_gemv(q, wd.k_pool, wd.v_pool, meta.block_tables, meta.kv_lens, n)
    want = call()
    torch.cuda.synchronize()
    recorder = _Recorder(_C._native)
    monkeypatch.setattr(_C, "_native", recorder)
    with torch.cuda.stream(torch.cuda.Stream()):
        _C._workspaces.pop((gpu.index, torch.cuda.current_stream(gpu).cuda_stream), None)
        first = call()
        torch.cuda.synchronize()
    for got in (first, call(q=q.as_subclass(Sub)), call(n=float(meta.max_kv_len))):
        assert torch.equal(got, want)
    assert recorder.declined == ["gemv"] * 3 and not recorder.took


def test_refused_calls_keep_their_errors(ops, gpu):
    from femtovllm import _C

    q = torch.zeros(4, 2, 128, dtype=torch.bfloat16, device=gpu)
    pool = torch.zeros(3, 2, 16, 128, dtype=torch.bfloat16, device=gpu)
    tables = torch.zeros(2, 2, dtype=torch.int32, device=gpu)
    lens = torch.ones(2, dtype=torch.int32, device=gpu)
    gemv = lambda **kw: ops.paged_attention_gemv(**{**dict(q=q, k_pool=pool, v_pool=pool, kv_page_tables=tables, kv_lens=lens, max_kv_len=32), **kw})
    gemv()
    for kw, text in [(dict(kv_lens=lens.long()), "kv_lens must be int32"), (dict(kv_page_tables=tables[:1]), "kv_page_tables.size"),
                     (dict(max_kv_len=8193), "kMaxKVLenNonSplit"), (dict(k_pool=pool.float()), "share a dtype"),
                     (dict(k_pool=pool[:, :1]), "contiguous"), (dict(kv_lens=lens.cpu()), "kv_lens must be on"),
                     (dict(q=q[:, :, :100]), "head_dim")]:
        with pytest.raises(RuntimeError, match=text):
            gemv(**kw)
    with pytest.raises(RuntimeError, match="q must be contiguous"):
        _C.PagedAttentionGemvCuda(torch.zeros(2, 4, 128, dtype=torch.bfloat16, device=gpu).transpose(0, 1), pool, pool, tables, lens, 32)
    with pytest.raises(RuntimeError, match="head_dim must be 128"):
        _C.FlashAttentionWarpCuda(*[torch.zeros(1, 2, 4, 64, dtype=torch.bfloat16, device=gpu)] * 3)
    with pytest.raises(RuntimeError):  # the library's own check: rows must be 16-byte aligned
        gemv(q=torch.zeros(4 * 2 * 128 + 1, dtype=torch.bfloat16, device=gpu)[1:].view(4, 2, 128))
