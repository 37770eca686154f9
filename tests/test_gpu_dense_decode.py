"""Decode over a page list (csrc/stream.hip) of batches: the dense decode, whose
split is made on the device from the page tables, and the layers of the shapes
without tuned kernels.

Dense outputs within 2e-3 of the fp64 softmax over the fp16 logits the
simulation rounds (quest_attention.py:265-268); a call's bits depend on its
sequences alone, not on the page count it was sized for.  A sequence of a
sparse layer's batch has the bits it has alone."""
import math
import sys

import pytest
import torch

from helpers import HND, NHD

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
I32 = dict(dtype=torch.int32, device=DEV)


@pytest.fixture(scope="module", autouse=True)
def _aoakv():
    import aoakv  # noqa: F401  (fails loudly if libaoakv.so is missing)
    yield


def _say(*a):
    print(*a, file=sys.stderr, flush=True)


class Batch:
    """K/V of sequences of these lengths in one paged cache: shuffled pages, a
    page table that starts 5 entries in, NaN in every unwritten slot."""

    def __init__(self, lens, D, S, H, hkv, layout=HND, seed=0):
        self.lens, self.D, self.S, self.H, self.hkv, self.layout = lens, D, S, H, hkv, layout
        g = torch.Generator(device=DEV).manual_seed(seed)
        self.P = [-(-n // S) for n in lens]
        total = sum(self.P)
        page = (2, S, hkv, D) if layout == NHD else (2, hkv, S, D)
        self.kv = torch.randn((total,) + page, generator=g, **dict(I32, dtype=torch.float16))
        self.indices = torch.cat([torch.zeros(5, **I32),
                                  torch.randperm(total, generator=g, device=DEV).int()])
        ptr = [5]
        for p in self.P:
            ptr.append(ptr[-1] + p)
        self.ptr = ptr
        self.indptr = torch.tensor(ptr, **I32)
        self.last = torch.tensor([(n - 1) % S + 1 for n in lens], **I32)
        tail = self.indices[self.indptr[1:].long() - 1].long()
        dead = torch.arange(S, device=DEV)[None] >= self.last[:, None]
        nhd = self.kv if layout == NHD else self.kv.transpose(2, 3)
        nhd[tail] = nhd[tail].masked_fill(dead[:, None, :, None, None], float("nan"))
        self.q = torch.randn((len(lens), H, D), generator=g, **dict(I32, dtype=torch.float16))

    def reference(self, b):
        x = self.kv[self.indices[self.ptr[b]:self.ptr[b + 1]].long()]
        x = (x if self.layout == NHD else x.transpose(2, 3)).transpose(0, 1)
        k, v = x.reshape(2, -1, self.hkv, self.D)[:, :self.lens[b]].double().transpose(1, 2)
        q = self.q[b].double().view(self.hkv, -1, self.D)
        logits = (torch.matmul(q, k.transpose(1, 2).contiguous()).half() /
                  math.sqrt(self.D)).half().double()
        return torch.matmul(torch.softmax(logits, -1), v.contiguous()).view(self.H, self.D)

    def dense(self, bound=None, flags=0, ws=None, runs=1):
        from aoakv import ops
        bound = bound or max(self.P)
        ws = ws if ws is not None else ops.decode_workspace(
            len(self.lens), self.H, self.hkv, bound, DEV, head_dim=self.D)
        for _ in range(runs):
            o = torch.full_like(self.q, float("nan"))
            ops.decode_sparse_attn(self.q, o, self.kv, self.indptr, self.indices, self.last, None,
                                   0, ws, bound, self.hkv, self.layout, flags=flags)
        assert int(ws.count_nonzero()) == 0  # no error, and all of it zero again
        return o


@pytest.mark.parametrize("H,hkv,D", [(32, 32, 128), (32, 8, 128), (16, 4, 128), (8, 8, 64),
                                     (16, 8, 256)])
@pytest.mark.parametrize("L", [1000, 2049, 3000, 5000, 16400])
def test_dense_bits_do_not_depend_on_the_bound(H, hkv, D, L):
    """The page count passed by value is the cache's capacity when a decode step
    is captured into a graph, and the sequence's own count otherwise."""
    from aoakv import ops
    _say(f"[dense bound] heads={H}/{hkv} D={D} L={L}")
    x = Batch([L], D, 16, H, hkv, seed=L)
    o = x.dense(runs=2)
    assert (o[0] - x.reference(0)).abs().max() <= 2e-3
    for bound in (x.P[0] + 1, 2048, 8192):
        assert torch.equal(x.dense(bound), o)
    if D == 128:
        assert torch.equal(x.dense(flags=ops.FLAG_GROUPED_DECODE), o)


# lengths: a few sequences (their share of the chunks), pages of one token,
# one long among short, one-page sequences between, as many as a wave has
# lanes and one more, and enough for a second and a third step of the search
BATCHES = [([1000, 999, 1001], 128, 16, 32, 8, HND), ([5, 1, 700], 64, 1, 4, 4, NHD),
           ([9000] + [17, 1, 300] * 5, 128, 16, 32, 32, HND),
           ([30000, 1, 16, 2000], 128, 16, 16, 4, NHD), ([40000, 64, 3], 64, 32, 8, 1, HND),
           ([50 + 7 * i for i in range(64)], 256, 7, 4, 2, HND),
           ([90 - i for i in range(65)], 128, 16, 8, 8, HND),
           ([3000] * 2 + [33] * 130 + [8000], 128, 8, 16, 2, NHD),
           ([1 + i % 40 for i in range(4200)], 64, 16, 2, 2, HND)]


@pytest.mark.parametrize("lens,D,S,H,hkv,layout", BATCHES)
def test_dense_batches(lens, D, S, H, hkv, layout):
    _say(f"[dense batch] {len(lens)} sequences up to {max(lens)} D={D} S={S} heads={H}/{hkv}")
    x = Batch(lens, D, S, H, hkv, layout, seed=len(lens))
    o = x.dense(runs=2)
    worst = max(float((o[b] - x.reference(b)).abs().max()) for b in range(len(lens)))
    assert worst <= 2e-3
    assert torch.equal(x.dense(max(x.P) * 3), o)


@pytest.mark.parametrize("lens,H,hkv", [([65536] + [1000] * 15, 32, 32),
                                        ([65536] + [1000] * 31, 32, 8)])
def test_a_long_sequence_of_a_batch_fills_the_chip(lens, H, hkv):
    """One long sequence among short ones takes about as long as as many tokens
    spread evenly (0.9 to 1.3 times; as one workgroup per head it took 4 to
    20 times as long)."""
    even = [sum(lens) // len(lens)] * len(lens)
    times = []
    for n in (lens, even):
        from aoakv import ops
        x = Batch(n, 128, 16, H, hkv)
        ws = ops.decode_workspace(len(n), H, hkv, max(x.P), DEV)
        x.dense(ws=ws, runs=3)
        best = float("inf")
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            o = torch.empty_like(x.q)
            a.record()
            for _ in range(10):
                ops.decode_sparse_attn(x.q, o, x.kv, x.indptr, x.indices, x.last, None, 0, ws,
                                       max(x.P), hkv, HND)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        times.append(best)
    _say(f"[dense ragged] heads={H}/{hkv} one long {times[0]:.0f} us, even {times[1]:.0f} us")
    assert times[0] < 2.5 * times[1]


@pytest.mark.parametrize("D,S,H,hkv,batch", [(64, 16, 4, 4, 1), (256, 16, 4, 2, 3),
                                             (128, 8, 8, 1, 70)])
def test_dense_page_tables_longer_than_the_bound(D, S, H, hkv, batch):
    """300 pages per table, sized for 200: the first 200 are attended, and flagged."""
    from aoakv import ops
    x = Batch([300 * S - 2] * batch, D, S, H, hkv, seed=3)
    ws = ops.decode_workspace(batch, H, hkv, 200, DEV, head_dim=D)
    o = torch.full_like(x.q, float("nan"))
    ops.decode_sparse_attn(x.q, o, x.kv, x.indptr, x.indices, x.last, None, 0, ws, 200, hkv, HND)
    assert ops.workspace_error(ws) == ops.WS_ERR_TRUNCATED
    assert int(ws.count_nonzero()) == 1  # the flag alone
    for b in range(batch):
        cut = Batch.__new__(Batch)
        cut.__dict__.update(x.__dict__)
        cut.ptr = [p for p in x.ptr]
        cut.ptr[b + 1] = cut.ptr[b] + 200
        cut.lens = [200 * S - 2] * batch
        assert (o[b] - cut.reference(b)).abs().max() <= 2e-3


def _layer(x, budgets, parts, bound, rows, flags):
    """sparse_decode_layer of the sequences `parts` of x; (o, sel, scores)."""
    from aoakv import ops
    B = len(parts)
    ptr, mptr, ids, mids = [0], [0], [], []
    for b in parts:
        ids.append(x.indices[x.ptr[b]:x.ptr[b + 1]])
        mids.append(x.m_indices[x.m_ptr[b]:x.m_ptr[b + 1]])
        ptr.append(ptr[-1] + ids[-1].numel())
        mptr.append(mptr[-1] + mids[-1].numel())
    q = x.q[parts].contiguous()
    o = torch.full_like(q, float("nan"))
    scores = torch.zeros((B, x.hkv, bound), dtype=torch.float32, device=DEV)
    sel = torch.full((B, x.hkv, rows), -1, **I32)
    ws = ops.decode_workspace(B, x.H, x.hkv, rows, DEV, max_pages=bound, head_dim=x.D)
    for _ in range(2):
        ops.sparse_decode_layer(q, o, x.kv, torch.tensor(ptr, **I32), torch.cat(ids), x.last[parts],
                                x.meta, torch.tensor(mptr, **I32), torch.cat(mids), x.lvn, scores,
                                sel, 0, ws, bound, x.layout, flags,
                                token_budgets=torch.tensor([budgets[b] for b in parts], **I32))
    return o, sel, scores, ws


def _with_metadata(x):
    """Appends every sequence's tokens again, with their page statistics."""
    from aoakv import ops
    pages, S = sum(x.P), x.S
    x.m_ptr = [0]
    for p in x.P:
        x.m_ptr.append(x.m_ptr[-1] + -(-p // S))
    x.m_indices = torch.randperm(x.m_ptr[-1], device=DEV).int()
    x.meta = torch.zeros((x.m_ptr[-1],) + tuple(x.kv.shape[1:]), dtype=torch.float16, device=DEV)
    x.lvn = torch.zeros((pages, x.hkv), dtype=torch.float16, device=DEV)
    mean = torch.zeros((pages, x.hkv, x.D), dtype=torch.float16, device=DEV)
    for b, n in enumerate(x.lens):
        ids = x.indices[x.ptr[b]:x.ptr[b + 1]]
        nhd = x.kv[ids.long()] if x.layout == NHD else x.kv[ids.long()].transpose(2, 3)
        k, v = nhd.transpose(0, 1).reshape(2, -1, x.hkv, x.D)[:, :n].contiguous()
        ops.append_kv_cache_prefill(k, v, x.kv, ids, x.P[b], (n - 1) % S + 1, x.meta,
                                    x.m_indices[x.m_ptr[b]:x.m_ptr[b + 1]], x.lvn, mean, x.layout)
    return x


@pytest.mark.parametrize("D,S,H,hkv,layout", [(64, 16, 8, 8, HND), (256, 16, 8, 4, NHD),
                                              (128, 8, 16, 4, HND), (128, 3, 4, 4, NHD)])
@pytest.mark.parametrize("batch", [6, 60])
def test_layer_of_a_ragged_batch_equals_its_sequences_alone(D, S, H, hkv, layout, batch):
    """Lengths from one token to 200 pages, budgets of their own; batches whose
    decode selects for itself and (60 sequences) that have a top-k launch."""
    from aoakv import ops
    _say(f"[ragged layer] D={D} S={S} heads={H}/{hkv} batch={batch}")
    lens = [(1, 200 * S, S, 37 * S + 2, 100 * S - 1, 9 * S)[b % 6] for b in range(batch)]
    x = _with_metadata(Batch(lens, D, S, H, hkv, layout, seed=D + S))
    budgets = [(S, 40 * S, 3 * S, 12 * S, 25 * S, 64 * S)[b % 6] for b in range(batch)]
    flags = ops.FLAG_VALUE_AWARE | ops.FLAG_FIXED
    o, sel, scores, ws = _layer(x, budgets, list(range(batch)), 200, 64, flags)
    assert int(ws.count_nonzero()) == 0
    assert torch.isfinite(o).all()
    for b in range(0, batch, 1 if batch < 10 else 7):
        P = x.P[b]
        k = min(max(3, min(lens[b], budgets[b]) // S), P)
        o1, sel1, scores1, _ = _layer(x, budgets, [b], P, max(3, k), flags)
        assert torch.equal(o[b], o1[0])
        assert torch.equal(sel[b, :, :k], sel1[0, :, :k]) and (sel[b, :, k:] == -1).all()
        assert torch.equal(scores[b, :, :P], scores1[0])


@pytest.mark.parametrize("D,S,H,hkv", [(64, 16, 4, 4), (256, 16, 4, 2), (128, 8, 32, 32)])
@pytest.mark.parametrize("batch", [1, 5])
def test_layer_of_page_tables_longer_than_the_bound(D, S, H, hkv, batch):
    """300 pages per table, sized for 200 (the decode selects for itself, or, of
    160 heads at 8 chunks, after a top-k launch): the bits of the 200-page
    tables, and the flag."""
    from aoakv import ops
    _say(f"[ragged layer, truncated] D={D} S={S} heads={H}/{hkv} batch={batch}")
    x = _with_metadata(Batch([300 * S - 2] * batch, D, S, H, hkv, seed=5))
    flags = ops.FLAG_VALUE_AWARE | ops.FLAG_FIXED
    budgets, parts = [64 * S] * batch, list(range(batch))
    got = _layer(x, budgets, parts, 200, 64, flags)
    assert ops.workspace_error(got[3]) == ops.WS_ERR_TRUNCATED
    assert int(got[3].count_nonzero()) == 1
    cut = Batch.__new__(Batch)
    cut.__dict__.update(x.__dict__)

    ids, mids = [], []
    for b in parts:
        ids.append(x.indices[x.ptr[b]:x.ptr[b] + 200])
        mids.append(x.m_indices[x.m_ptr[b]:x.m_ptr[b] + -(-200 // S)])
    cut.indices, cut.m_indices = torch.cat(ids), torch.cat(mids)
    cut.ptr = [200 * b for b in range(batch + 1)]
    cut.m_ptr = [-(-200 // S) * b for b in range(batch + 1)]
    want = _layer(cut, budgets, parts, 200, 64, flags)
    assert ops.workspace_error(want[3]) == 0
    for a, b in zip(got[:3], want[:3]):
        assert torch.equal(a, b)
