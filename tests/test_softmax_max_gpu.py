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
