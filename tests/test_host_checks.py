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


def _valid():
    """entry point -> (argument names, arguments of a call that runs): one
    sequence of 19 tokens, 4 kv heads of 128 in pages of 16 (HND), 8 query
    heads; 2 pages, one of them selectable."""
    d = "cuda:0"
    z = lambda *s: torch.zeros(s, dtype=H, device=d)
    i = lambda *v: torch.tensor(v, dtype=I, device=d)
    t = dict(kv_data=z(2, 2, 4, 16, 128), metadata_data=z(1, 2, 4, 16, 128), v_log_norm=z(2, 4),
             v_mean=z(2, 4, 128), kv_indptr=i(0, 2), kv_indices=i(1, 0), kv_last_page_len=i(3),
             metadata_indptr=i(0, 1), metadata_indices=i(0), k=z(1, 4, 128), v=z(1, 4, 128),
             q=z(1, 8, 128), o=z(1, 8, 128), scores=torch.zeros((1, 4, 2), device=d),
             sel_pages=torch.zeros((1, 4, 3), dtype=I, device=d), token_budget=32,
             token_budgets=i(32), workspace=ops.decode_workspace(1, 8, 4, 3, d, max_pages=2),
             max_pages=2, num_kv_heads=4, page_size=16, layout=1, num_kv_pages=2, last=3,
             flags=ops.FLAG_VALUE_AWARE | ops.FLAG_FIXED, x=z(3, 64), weight=z(64), out=z(3, 64),
             eps=1e-6, causal=True, input=z(3, 64), output=z(3, 64))
    cache = "metadata_data metadata_indices v_log_norm v_mean layout"
    batch = "kv_data kv_indptr kv_indices kv_last_page_len metadata_data metadata_indptr " \
            "metadata_indices v_log_norm v_mean layout"
    names = {
        "append_kv_cache_prefill": "k v kv_data kv_indices num_kv_pages last " + cache,
        "append_kv_cache_decode": "k v " + batch,
        "rope_append_kv_cache_prefill": "q k v kv_data kv_indices num_kv_pages last " + cache,
        "rope_append_kv_cache_decode": "q k v " + batch,
        "estimate_attn_score": "q scores metadata_data metadata_indptr metadata_indices kv_indptr "
                               "kv_indices kv_last_page_len v_log_norm max_pages layout",
        "topk_filtering": "scores kv_indptr kv_indices kv_last_page_len token_budget sel_pages "
                          "page_size flags token_budgets workspace",
        "decode_sparse_attn": "q o kv_data kv_indptr kv_indices kv_last_page_len sel_pages "
                              "token_budget workspace max_pages num_kv_heads layout token_budgets",
        "sparse_decode_layer": "q o kv_data kv_indptr kv_indices kv_last_page_len metadata_data "
                               "metadata_indptr metadata_indices v_log_norm scores sel_pages "
                               "token_budget workspace max_pages layout flags token_budgets",
        "prefill_with_paged_kv_cache": "q kv_data kv_indices num_kv_pages last layout causal o",
        "rms_norm_forward": "input weight output eps",
    }
    return {f: (n.split(), [t[x] for x in n.split()]) for f, n in names.items()}


# (entry points, argument, what becomes of it, error, message)
APPENDS = ["append_kv_cache_prefill", "append_kv_cache_decode", "rope_append_kv_cache_prefill",
           "rope_append_kv_cache_decode"]
DECODES = ["append_kv_cache_decode", "rope_append_kv_cache_decode"]
PREFILLS = ["append_kv_cache_prefill", "rope_append_kv_cache_prefill"]
CACHES = APPENDS + ["decode_sparse_attn", "sparse_decode_layer", "prefill_with_paged_kv_cache"]
BREAKS = [
    (CACHES, "kv_data", lambda t: t[0], ValueError, "paged cache must be 5-d"),
    (CACHES, "kv_data", lambda t: t[:, :1].contiguous(), ValueError, "paged cache must be 5-d"),
    (["estimate_attn_score"], "metadata_data", lambda t: t[0], ValueError,
     "paged cache must be 5-d"),
    (CACHES + ["estimate_attn_score"], "layout", lambda x: 2, ValueError, "unknown layout 2"),
    (PREFILLS, "k", lambda t: t[:, :3].contiguous(), ValueError, r"k/v must be \[N, 4, 128\], got"),
    (PREFILLS, "v", lambda t: t.repeat(2, 1, 1), ValueError, r"k/v must be \[N, 4, 128\], got"),
    (PREFILLS, "kv_indices", lambda t: t[:1].clone(), ValueError, "kv_indices shorter"),
    (PREFILLS, "last", lambda x: 17, RuntimeError, "kv_last_page_len 17 not in"),
    (["rope_append_kv_cache_prefill"], "q", lambda t: t.repeat(2, 1, 1), ValueError, "q must be"),
    (DECODES, "k", lambda t: t[..., :64].contiguous(), ValueError, "k/v (must be )?.?.?B, 4, 128"),
    (DECODES, "v", lambda t: t.repeat(2, 1, 1), ValueError, "k/v"),
    (["rope_append_kv_cache_decode"], "q", lambda t: t[0], ValueError, "q must be"),
    (["rope_append_kv_cache_decode"], "q", lambda t: t[..., :64].contiguous(), ValueError,
     "q must be"),
    (DECODES, "kv_indptr", lambda t: t[:1].clone(), ValueError, "sizes do not match the batch"),
    (DECODES, "kv_last_page_len", lambda t: t.repeat(2), ValueError,
     "sizes do not match the batch"),
    (DECODES, "metadata_indptr", lambda t: t.repeat(2), ValueError,
     "sizes do not match the batch"),
    (["estimate_attn_score", "decode_sparse_attn", "sparse_decode_layer"], "q", lambda t: t[0],
     ValueError, r"q must be \[B, Hq, D\]"),
    (["estimate_attn_score"], "q", lambda t: t[..., :64].contiguous(), ValueError,
     "scores must be"),
    (["estimate_attn_score"], "scores", lambda t: t[0], ValueError, "scores must be"),
    (["estimate_attn_score"], "scores", lambda t: t.repeat(2, 1, 1), ValueError,
     "scores must be"),
    (["estimate_attn_score"], "scores", lambda t: t[:, :3].contiguous(), ValueError,
     "scores must be"),
    (["estimate_attn_score"], "scores", lambda t: t[..., :1].contiguous(), RuntimeError,
     "score_stride"),
    (["topk_filtering"], "scores", lambda t: t[0], ValueError, "scores must be"),
    (["topk_filtering"], "sel_pages", lambda t: t[0], ValueError, "sel_pages must be"),
    (["topk_filtering"], "sel_pages", lambda t: t[:, :3].contiguous(), ValueError,
     "sel_pages must be"),
    (["topk_filtering"], "workspace", lambda t: t[:8].clone(), ValueError, "workspace too small"),
    (["topk_filtering", "decode_sparse_attn", "sparse_decode_layer"], "token_budgets",
     lambda t: t.long(), TypeError, "token_budgets must be torch.int32, got torch.int64"),
    (["decode_sparse_attn"], "o", lambda t: t[:, :4].contiguous(), ValueError, "o must have q's"),
    (["decode_sparse_attn"], "num_kv_heads", lambda x: 8, ValueError, "num_kv_heads does not match"),
    (["decode_sparse_attn"], "sel_pages", lambda t: t.float(), TypeError,
     "sel_pages must be torch.int32"),
    (["decode_sparse_attn", "sparse_decode_layer"], "workspace", lambda t: t[:256].clone(),
     RuntimeError, "workspace of 256 bytes"),
    (["sparse_decode_layer"], "scores", lambda t: t[0, 0, 0], ValueError, "must have rows"),
    (["sparse_decode_layer"], "sel_pages", lambda t: t[0, 0, 0], ValueError, "must have rows"),
    (["sparse_decode_layer"], "sel_pages", lambda t: t[..., :2].contiguous(), RuntimeError,
     "sel_stride 2 < 3"),
    (["estimate_attn_score", "sparse_decode_layer"], "v_log_norm", lambda t: None, TypeError,
     "v_log_norm must be a torch.Tensor"),
    (["sparse_decode_layer"], "kv_indptr", lambda t: None, AttributeError, "page table"),
    (["prefill_with_paged_kv_cache"], "q", lambda t: t[0], ValueError, "q must be"),
    (["prefill_with_paged_kv_cache"], "q", lambda t: t[..., :64].contiguous(), ValueError,
     "q must be"),
    (["prefill_with_paged_kv_cache"], "q", lambda t: t[:, :0].contiguous(), RuntimeError,
     "num_heads 0"),
    (["prefill_with_paged_kv_cache"], "q", lambda t: t.repeat(20, 1, 1), RuntimeError,
     "qo_len 20 not in"),
    (["prefill_with_paged_kv_cache"], "o", lambda t: "x", TypeError, "o must be a torch.Tensor"),
    (["rms_norm_forward"], "weight", lambda t: t[:32].clone(), ValueError,
     r"weight must be \[64\]"),
    (["rms_norm_forward"], "output", lambda t: t[:2].clone(), ValueError, r"output \(3, 64\)"),
    (["rms_norm_forward"], "input", lambda t: t[0, 0], ValueError, "last dimension"),
]
CASES = [(f, *b[1:]) for b in BREAKS for f in b[0]]


@pytest.mark.gpu
def test_valid_calls_run():
    for f, (_, args) in _valid().items():
        getattr(ops, f)(*args)
    torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("name,arg,change,error,message", CASES,
                         ids=[f"{c[0]}-{c[1]}-{n}" for n, c in enumerate(CASES)])
def test_one_wrong_argument_is_named(name, arg, change, error, message):
    """A call that runs with one argument changed: that argument's own check."""
    names, args = _valid()[name]
    args[names.index(arg)] = change(args[names.index(arg)])
    with pytest.raises(error, match=message):
        getattr(ops, name)(*args)
