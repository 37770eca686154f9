"""The checks of the C++ tensor wrappers (aoakv._host) raise what the Python
wrappers of the other entry points raise, before anything is launched."""
import ctypes

import pytest
import torch

from aoakv import ops

# entry point -> its arguments, a tensor as its dtype
H, I, F, B = torch.float16, torch.int32, torch.float32, torch.uint8
CALLS = {
    "append_kv_cache_prefill": [H, H, H, I, 1, 1, H, I, H, H, 1],
    "append_kv_cache_decode": [H, H, H, I, I, I, H, I, I, H, H, 1],
    "rope_append_kv_cache_decode": [H, H, H, H, I, I, I, H, I, I, H, H, 1],
    "rope_append_kv_cache_prefill": [H, H, H, H, I, 1, 1, H, I, H, H, 1],
    "estimate_attn_score": [H, F, H, I, I, I, I, I, H, 1, 1],
    "topk_filtering": [F, I, I, I, 64, I],
    "decode_sparse_attn": [H, H, H, I, I, I, I, 64, B, 1, 1, 1],
    "sparse_decode_layer": [H, H, H, I, I, I, H, I, I, H, F, I, 64, B, 1, 1],
    "prefill_with_paged_kv_cache": [H, H, I, 1, 1, 1],
    "rms_norm_forward": [H, H, H, 1e-6],
}


def _args(spec, device="cpu"):
    return [torch.zeros(4, dtype=x, device=device) if isinstance(x, torch.dtype) else x
            for x in spec]


@pytest.mark.parametrize("name", CALLS)
def test_types_and_devices(name):
    f, spec = getattr(ops, name), CALLS[name]
    with pytest.raises(ValueError, match="must be a device tensor"):
        f(*_args(spec))
    bad = _args(spec)
    bad[0] = "x"
    with pytest.raises(TypeError, match="must be a torch.Tensor"):
        f(*bad)
    bad[0] = torch.zeros(4, dtype=torch.float64)
    with pytest.raises(TypeError, match="must be torch.float(16|32), got torch.float64"):
        f(*bad)


@pytest.mark.gpu
@pytest.mark.parametrize("name", CALLS)
def test_shapes_and_layout(name):
    f, spec = getattr(ops, name), CALLS[name]
    args = _args(spec, "cuda:0")
    with pytest.raises((ValueError, ops._lib.AoakvError)):  # 1-d tensors everywhere
        f(*args)
    args[0] = torch.zeros((4, 4, 2), dtype=spec[0], device="cuda:0").transpose(0, 1)
    with pytest.raises(ValueError, match="must be contiguous"):
        f(*args)


@pytest.mark.gpu
def test_integers_layout_and_status():
    z = lambda *s: torch.zeros(s, dtype=H, device="cuda:0")
    i = lambda *s: torch.zeros(s, dtype=I, device="cuda:0")
    cache, k = z(2, 2, 4, 16, 128), z(3, 4, 128)
    rest = (z(1, 2, 4, 16, 128), i(1), z(2, 4), z(2, 4, 128))
    with pytest.raises(ctypes.ArgumentError):
        ops.append_kv_cache_prefill(k, k, cache, i(2), 1.0, 3, *rest, 1)
    with pytest.raises(ValueError, match="unknown layout 2"):
        ops.append_kv_cache_prefill(k, k, cache, i(2), 1, 3, *rest, 2)
    with pytest.raises(ValueError, match="kv_indices shorter"):
        ops.append_kv_cache_prefill(k, k, cache, i(2), 3, 3, *rest, 1)
    with pytest.raises(ValueError, match=r"k/v must be \[N, 4, 128\], got \(3, 4, 128\) / \(2, 4, 128\)"):
        ops.append_kv_cache_prefill(k, z(2, 4, 128), cache, i(2), 1, 3, *rest, 1)
    with pytest.raises(ops._lib.AoakvError, match="3 new tokens but the cache holds 2") as e:
        ops.append_kv_cache_prefill(k, k, cache, i(2), 1, 2, *rest, 1)
    assert e.value.code == ops._lib.AOAKV_ERR_INVALID


@pytest.mark.gpu
def test_integers_are_compared_whole():
    """Arguments that are checked against a tensor's size (and the layout) are
    not cut to 32 bits first, and the kv head count may be any number type;
    a value statistic is a tensor whether the flags use it or not."""
    import numpy as np
    z = lambda *s: torch.zeros(s, dtype=H, device="cuda:0")
    i = lambda *s: torch.zeros(s, dtype=I, device="cuda:0")
    cache, k = z(2, 2, 4, 16, 128), z(3, 4, 128)
    rest = (z(1, 2, 4, 16, 128), i(1), z(2, 4), z(2, 4, 128))
    for pages in (2**32 + 1, 2**64 + 1, -1):
        with pytest.raises(ValueError, match="kv_indices shorter"):
            ops.append_kv_cache_prefill(k, k, cache, i(2), pages, 3, *rest, 1)
        with pytest.raises(ValueError, match="kv_indices shorter"):
            ops.rope_append_kv_cache_prefill(k.clone(), k.clone(), k, cache, i(2), pages, 3, *rest, 1)
    for layout in (2**32 + 1, -1, 2**80):
        with pytest.raises(ValueError, match=f"unknown layout {layout}"):
            ops.append_kv_cache_prefill(k, k, cache, i(2), 1, 3, *rest, layout)
    q, ip, last = z(1, 4, 128), torch.tensor([0, 1], **dict(dtype=I, device="cuda:0")), i(1) + 3
    ws = ops.decode_workspace(1, 4, 4, 2, "cuda:0")
    for heads in (np.int64(4), 4.0):
        o = torch.full_like(q, float("nan"))
        ops.decode_sparse_attn(q, o, cache, ip, i(2), last, None, 0, ws, 2, heads, 1)
        assert torch.equal(o, torch.zeros_like(o))
    for heads in (3, 2**32 + 4):
        with pytest.raises(ValueError, match="num_kv_heads does not match"):
            ops.decode_sparse_attn(q, o, cache, ip, i(2), last, None, 0, ws, 2, heads, 1)
    scores = torch.zeros((1, 4, 2), device="cuda:0")
    with pytest.raises(AttributeError):
        ops.estimate_attn_score(q, scores, rest[0], ip, i(1), ip, i(2), last, "x", 2, 1, 0)
    with pytest.raises(AttributeError):
        ops.sparse_decode_layer(q, o, cache, ip, i(2), last, rest[0], ip, i(1), "x", scores,
                                i(1, 4, 3), 32, ws, 2, 1, 0)
