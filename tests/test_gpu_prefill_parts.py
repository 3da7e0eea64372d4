"""Global prefill chunks of few row blocks run their key tiles in parts on
several workgroups, which merge them through the workspace: the edges of row
blocks, tiles and parts, ragged batches, unmapped pages, smaller workspaces, a
balanced chunk on the same workspace afterwards, other work on the GPU."""
import ctypes
import math

import numpy as np
import pytest

import gemma_kv as gk
from kvtest import assert_close, cache_config, empty_bf16, fill_page_table, from_dev_bf16, randn_bf16, to_dev
from oracle import oracle

pytestmark = pytest.mark.gpu
H, D = 8, 256
SLOT_BYTES = 256 + 2 * 130 * 256 * 4


def _run(dev, priors, lq, page, ws=None, ws_bytes=None, capacity=0):
    import torch
    rng = np.random.default_rng(lq * 7 + sum(priors))
    batch = len(priors)
    max_pages = max(capacity, max(priors) + lq) // page + 1
    cfg = cache_config(1, batch, page, max_pages, H, D, 0)
    pt = fill_page_table(cfg, priors)
    q = randn_bf16(rng, (batch, lq, 16, D))
    k, v = randn_bf16(rng, (batch, lq, H, D)), randn_bf16(rng, (batch, lq, H, D))
    ck, cv = (randn_bf16(rng, (batch * max_pages * page, H, D)) for _ in range(2))
    c = gk.make_config(*cfg)
    need = gk.flash_attention_prefill_chunk_workspace_bytes(batch, lq, c)
    if ws is None:
        ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    args = [to_dev(x, dev) for x in (q, k, v, ck, cv, pt, np.asarray(priors, np.int32))]
    scale = 1 / math.sqrt(D)
    out, plain = empty_bf16((batch, lq, 16, D), dev), empty_bf16((batch, lq, 16, D), dev)
    print(f"priors {priors} rows {lq} page {page} workspace {ws_bytes or ws.numel()}", flush=True)
    gk.check(gk.flash_attention_prefill_chunk_paged_bf16_ws(
        out, *args, c, 0, batch, lq, scale, ws, ws_bytes or ws.numel()))
    gk.check(gk.flash_attention_prefill_chunk_paged_bf16(plain, *args, c, 0, batch, lq, scale))
    torch.cuda.synchronize()
    got = from_dev_bf16(out)
    assert_close(got, from_dev_bf16(plain), f"parts vs plain {priors} {lq}")
    rows = pt.reshape(batch, max_pages).astype(np.int64)
    b = batch - 1
    pos = np.arange(priors[b])
    r = rows[b, pos // page] * page + pos % page
    full = [np.concatenate([c0[r], new[b]])[None] for c0, new in ((ck, k), (cv, v))]
    exp = oracle.prefill_attention(q[b:b + 1], *full, lq, priors[b] + lq, 16, H, D, 0, scale)[0]
    assert_close(got[b], exp, f"parts vs oracle {priors} {lq}")
    return ws


@pytest.mark.parametrize("priors,lq,page", [
    ([500], 1, 16),            # one row, one row block: eight parts of 32
    ([0], 64, 16),             # a single part: its workgroup writes the rows
    ([128 - 64], 64, 16),      # two tiles
    ([129 - 64], 64, 64),      # three tiles
    ([2047], 1, 16),           # 32 tiles for 32 parts
    ([2048], 1, 16),           # 33: 17 parts, the last of one tile
    ([900], 63, 1),
    ([700], 65, 16),           # the second row block holds one row
    ([3, 1200, 400], 17, 16),  # ragged: one, several and many parts
    ([100], 400, 16),          # parts of the chunk's own keys
    ([37], 1000, 16),          # two parts per row block
])
def test_parts_match_oracle(dev, priors, lq, page):
    _run(dev, priors, lq, page, capacity=512)


def test_parts_and_balanced_chunks_share_a_workspace(dev):
    ws = _run(dev, [600], 40, 16)
    ws = _run(dev, [9], 1100, 16, ws)    # 18 row blocks: balanced
    ws = _run(dev, [600], 40, 16, ws)
    assert not ws[: ws.numel() // SLOT_BYTES * SLOT_BYTES].view(-1, SLOT_BYTES)[:, :4].any().item()


@pytest.mark.parametrize("slots", [0, 3, 8, 20])
def test_smaller_workspaces_stay_accepted(dev, slots):
    """A single row block needs no workspace; what there is gives fewer parts."""
    import torch
    ws = torch.zeros(max(slots, 1) * SLOT_BYTES, dtype=torch.uint8, device=dev)
    _run(dev, [700], 50, 16, ws, max(1, slots * SLOT_BYTES))


def test_workspace_bytes_never_shrink_with_the_call():
    c = gk.make_config(*cache_config(1, 4, 64, 64, H, D, 0))
    largest = gk.flash_attention_prefill_chunk_workspace_bytes(4, 2048, c)
    for n in (1, 64, 65, 512, 1024, 1025, 2048):
        sizes = [gk.flash_attention_prefill_chunk_workspace_bytes(b, n, c) for b in (1, 2, 4)]
        assert sizes == sorted(sizes) and sizes[-1] <= largest


@pytest.mark.parametrize("prior,lq", [(600, 40), (129, 64), (1537, 100)])
def test_infinite_values(dev, prior, lq):
    """An infinite V element of the last cached key, which every row sees, in
    the last part of a row block: infinite in that dim, finite and right
    elsewhere."""
    import torch
    rng = np.random.default_rng(prior)
    page = 16
    max_pages = (prior + lq) // page + 1
    cfg = cache_config(1, 1, page, max_pages, H, D, 0)
    q, k, v = (randn_bf16(rng, (1, lq, h, D)) for h in (16, H, H))
    ck, cv = (randn_bf16(rng, (max_pages * page, H, D)) for _ in range(2))
    pt = fill_page_table(cfg, [prior])
    pos = np.arange(prior)
    r = pt[pos // page].astype(np.int64) * page + pos % page
    cv[r[-1], :, 7], cv[r[-1], :, 250] = 0x7F80, 0xFF80
    c = gk.make_config(*cfg)
    need = gk.flash_attention_prefill_chunk_workspace_bytes(1, lq, c)
    ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    out = empty_bf16((1, lq, 16, D), dev)
    gk.check(gk.flash_attention_prefill_chunk_paged_bf16_ws(
        out, *(to_dev(x, dev) for x in (q, k, v, ck, cv, pt, np.int32([prior]))), c, 0, 1, lq, 1 / 16, ws, need))
    torch.cuda.synchronize()
    got = from_dev_bf16(out)
    finite = np.where((cv & 0x7FFF) == 0x7F80, 0, cv)
    full = [np.concatenate([c0[r], new[0]])[None] for c0, new in ((ck, k), (finite, v))]
    exp = oracle.prefill_attention(q, *full, lq, prior + lq, 16, H, D, 0, 1 / 16)
    assert (got[..., 7] == 0x7F80).all() and (got[..., 250] == 0xFF80).all()
    rest = [d for d in range(D) if d not in (7, 250)]
    assert_close(got[..., rest], exp[..., rest], "finite dims")


class _Call:
    """A chunk of `lq` rows after `prior` keys for each sequence, on the GPU, bound to its workspace."""

    def __init__(self, dev, prior, lq, capacity=8192, hole=None, batch=1):
        import torch
        gen = torch.Generator(device=dev).manual_seed(prior + lq)

        def rnd(*shape):
            return torch.randn(shape, generator=gen, device=dev, dtype=torch.bfloat16)
        cfg = cache_config(1, batch, 64, capacity // 64, H, D, 0)
        table = np.arange(batch * (capacity // 64), dtype=np.int32)
        if hole is not None:
            table[hole] = -1
        self.c = gk.make_config(*cfg)
        rows = batch * capacity
        self.args = [rnd(batch, lq, 16, D), rnd(batch, lq, H, D), rnd(batch, lq, H, D), rnd(rows, H, D), rnd(rows, H, D),
                     to_dev(table, dev), torch.tensor([prior] * batch, dtype=torch.int32, device=dev)]
        self.batch, self.lq = batch, lq
        need = gk.flash_attention_prefill_chunk_workspace_bytes(batch, lq, self.c)
        self.ws = torch.zeros(need, dtype=torch.uint8, device=dev)

    def plain(self):
        import torch
        out = torch.empty_like(self.args[0])
        gk.check(gk.flash_attention_prefill_chunk_paged_bf16(out, *self.args, self.c, 0, self.batch, self.lq, 1 / 16))
        return out

    def parts(self, out=None):
        import torch
        out = torch.full_like(self.args[0], float("nan")) if out is None else out
        gk.check(gk.flash_attention_prefill_chunk_paged_bf16_ws(
            out, *self.args, self.c, 0, self.batch, self.lq, 1 / 16, self.ws, self.ws.numel()))
        return out

    def counters_are_zero(self):
        return not self.ws.view(-1, SLOT_BYTES)[:, :256].any().item()


def _close(a, b, what):
    import torch
    assert_close(*(from_dev_bf16(x.view(torch.int16)) for x in (a, b)), what)


def test_a_chunk_is_one_launch(dev):
    """In parts or not, with keys to share out or not: the host cannot know,
    and a second launch would be paid for by short chunks as well."""
    import torch
    hip = ctypes.CDLL("libamdhip64.so.7")
    for prior, lq in ((0, 64), (2000, 64), (0, 1100)):
        call = _Call(dev, prior, lq)
        out = call.parts()
        torch.cuda.synchronize()
        stream, graph, nodes = torch.cuda.Stream(), ctypes.c_void_p(), ctypes.c_size_t()
        handle = ctypes.c_void_p(stream.cuda_stream)
        with torch.cuda.stream(stream):
            assert hip.hipStreamBeginCapture(handle, 2) == 0  # relaxed
            call.parts(out)
            assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
        assert nodes.value == 1, (prior, lq)
        assert hip.hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("prior,lq,hole", [(1000, 33, 3), (1000, 33, 15), (200, 100, 1), (5000, 1, 70)])
def test_parts_over_unmapped_pages(dev, prior, lq, hole):
    """A part without a readable key (a part is one 64-key tile in the first
    three, as a page is), among them the last cached page; one tile of three."""
    call = _Call(dev, prior, lq, hole=hole)
    _close(call.parts(), call.plain(), f"hole {hole}")
    assert call.counters_are_zero()


def test_parts_repeat_bit_for_bit_beside_other_work(dev):
    """Who merges depends on when the workgroups run; the bits do not. Calls
    beside matrix products that fill the GPU, and on replays of a graph."""
    import torch
    x = torch.randn(4096, 4096, device=dev).bfloat16()
    other = torch.cuda.Stream()
    for prior, lq in ((130, 64), (7401, 93), (3000, 1), (900, 300), (400, 1000)):
        call = _Call(dev, prior, lq)
        print(f"prior {prior} rows {lq}", flush=True)
        first = call.parts()
        _close(first, call.plain(), "alone")
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            for _ in range(20):
                x @ x
        outs = [call.parts() for _ in range(25)]
        torch.cuda.synchronize()
        assert all(torch.equal(o, first) for o in outs)
        assert call.counters_are_zero()
        out, graph = torch.empty_like(first), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call.parts(out)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, first)


def test_long_parts(dev):
    """31 parts of 39 tiles and one of 40."""
    call = _Call(dev, 1248 * 64, 64, capacity=1249 * 64)
    _close(call.parts(), call.plain(), "long")
    assert call.counters_are_zero()


@pytest.mark.parametrize("batch,prior,lq,shared", [
    (1, 0, 64, False),       # one tile
    (1, 37, 64, True),       # two
    (4, 0, 64, False), (16, 64, 64, False), (16, 1200, 64, True),
    (8, 100, 128, False), (8, 900, 128, True),
    (2, 100, 300, True),     # row blocks of one part and of more
    (1, 0, 1000, True), (5, 800, 192, True), (1, 4000, 1, True),
])
def test_row_blocks_are_shared_out_where_it_pays(dev, batch, prior, lq, shared):
    """Partials are written for enough keys per row and not otherwise: of many
    short row blocks they cost more than the shorter chains save."""
    call = _Call(dev, prior, lq, capacity=4096, batch=batch)
    out = call.parts()
    assert call.ws.any().item() == shared
    _close(out, call.plain(), "parts")
    assert call.counters_are_zero()
