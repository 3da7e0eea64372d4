"""The 1 x 512 split kernel (decode_d512.hip) against the oracle at the sizes
where it can go wrong: splits of one key to several steps of both workgroup
forms (a step is 16 keys per wave), ragged last tiles, idle waves, page
lookups past the first four steps, rings, unmapped pages, and batches whose
splits the device cuts by the lengths (more planned splits than workgroups).
Cache rows that no sequence may read hold NaN: a value that leaks through a
masked key shows."""
import math

import numpy as np
import pytest

import gemma_kv as gk
from kvtest import assert_close, cache_config, fill_page_table, from_dev_bf16, randn_bf16, ring_pages, to_dev
from oracle import oracle
from test_gpu_decode import _run_decode
from test_gpu_decode_prep import _close_bits

pytestmark = pytest.mark.gpu
NAN = np.uint16(0x7FC0)

# (split size, lengths, window, page)
CASES = [
    (1, [3], 0, 16),
    (15, [31], 0, 16),
    (16, [33], 0, 1),
    (48, [8, 97], 0, 16),              # cut by length: 2 x 3 slots, all run
    (63, [64, 127, 190], 0, 64),
    (64, [1, 64, 65], 0, 16),
    (65, [66], 0, 16),                 # two-wave form: a step and one key
    (96, [95, 96, 97, 0, 300], 0, 64),
    (160, [159, 161], 0, 16),          # past four steps: the second page lookup
    (333, [1000], 0, 16),
    (512, [512], 0, 64),               # a single split, written directly
    (40, [500], 256, 16),              # a ring, split by position
    (70, [80, 256, 700], 256, 1),
    (16, [4001, 17, 2900], 0, 64),     # 753 planned splits on 512 workgroups
    (16, [11 * i for i in range(64)], 0, 16),
    (16, [9 * i for i in range(65)], 0, 16),  # past the batch that is cut by length
]


def _case(rng, split, seq, window, page):
    batch = len(seq)
    max_pages = ring_pages(window, page) if window else max(1, -(-max(seq) // page))
    cfg = cache_config(1, batch, page, max_pages, 1, 512, window)
    pt = fill_page_table(cfg, seq)
    rows = batch * max_pages * page
    ck, cv = np.full((rows, 1, 512), NAN), np.full((rows, 1, 512), NAN)
    for b, n in enumerate(seq):
        pos = np.arange(max(0, n - window) if window else 0, n)
        r = pt[b * max_pages + (pos // page) % max_pages].astype(np.int64) * page + pos % page
        ck[r], cv[r] = randn_bf16(rng, (len(r), 1, 512)), randn_bf16(rng, (len(r), 1, 512))
    live = max(min(n, window) if window else n for n in seq)
    return cfg, pt, ck, cv, randn_bf16(rng, (batch, 16, 512)), -(-live // split)


@pytest.mark.parametrize("split,seq,window,page", CASES)
def test_split_sizes(dev, split, seq, window, page):
    rng = np.random.default_rng(split * 1000 + len(seq))
    cfg, pt, ck0, cv0, q, splits = _case(rng, split, seq, window, page)
    print(f"split {split}x{splits} seq {seq[:6]} window {window} page {page}", flush=True)
    scale = 1.0 / math.sqrt(512)
    # The token of the last position; a sequence without keys has none.
    k, v = randn_bf16(rng, (len(seq), 1, 512)), randn_bf16(rng, (len(seq), 1, 512))
    pos = [n - 1 for n in seq]
    exp_k, exp_v = ck0.copy(), cv0.copy()
    oracle.kv_cache_write(exp_k, exp_v, cfg, pt, list(range(len(seq))), pos, 0, k, v)
    exp = oracle.decode_attention(q, exp_k, exp_v, pt, seq, cfg, 0, scale)
    ck, cv = to_dev(ck0, dev), to_dev(cv0, dev)
    got = _run_decode(dev, cfg, q, ck, cv, pt, seq, 0, scale, split, splits, fused=(pos, k, v))
    assert np.array_equal(from_dev_bf16(ck).reshape(exp_k.shape), exp_k)
    assert np.array_equal(from_dev_bf16(cv).reshape(exp_v.shape), exp_v)
    assert_close(got, exp, "appended")
    # The same without an append, over the cache it left.
    got = _run_decode(dev, cfg, q, ck, cv, pt, seq, 0, scale, split, splits)
    assert_close(got, exp, "no append")


def test_unmapped_pages_in_a_batch(dev):
    """Unmapped pages inside the live range, among them the token's own."""
    rng = np.random.default_rng(77)
    seq = [200, 90, 333]
    cfg, pt, ck0, cv0, q, splits = _case(rng, 16, seq, 0, 16)
    max_pages = cfg[3]
    pt[3] = pt[max_pages + 5] = pt[2 * max_pages + 20] = -1  # page 5 holds position 89
    k, v = randn_bf16(rng, (3, 1, 512)), randn_bf16(rng, (3, 1, 512))
    pos = [n - 1 for n in seq]
    exp_k, exp_v = ck0.copy(), cv0.copy()
    oracle.kv_cache_write(exp_k, exp_v, cfg, pt, [0, 1, 2], pos, 0, k, v)
    exp = oracle.decode_attention(q, exp_k, exp_v, pt, seq, cfg, 0, 0.0442)
    ck, cv = to_dev(ck0, dev), to_dev(cv0, dev)
    got = _run_decode(dev, cfg, q, ck, cv, pt, seq, 0, 0.0442, 16, splits, fused=(pos, k, v))
    assert np.array_equal(from_dev_bf16(ck).reshape(exp_k.shape), exp_k)
    assert_close(got, exp, "unmapped")


def test_token_outside_the_live_keys_is_appended(dev):
    """A token past its sequence's length (also an empty one) is stored and
    not attended to, in a batch cut by its lengths."""
    rng = np.random.default_rng(78)
    held = [40, 16, 600]
    cfg, pt, ck0, cv0, q, _ = _case(rng, 16, held, 0, 16)
    seq = [20, 0, 599]
    k, v = randn_bf16(rng, (3, 1, 512)), randn_bf16(rng, (3, 1, 512))
    pos = [33, 4, 599]
    exp = oracle.decode_attention(q, ck0, cv0, pt, seq, cfg, 0, 0.05)
    exp_k, exp_v = ck0.copy(), cv0.copy()
    oracle.kv_cache_write(exp_k, exp_v, cfg, pt, [0, 1, 2], pos, 0, k, v)
    ck, cv = to_dev(ck0, dev), to_dev(cv0, dev)
    got = _run_decode(dev, cfg, q, ck, cv, pt, seq, 0, 0.05, 16, 38, fused=(pos, k, v))
    assert np.array_equal(from_dev_bf16(ck).reshape(exp_k.shape), exp_k)
    assert np.array_equal(from_dev_bf16(cv).reshape(exp_v.shape), exp_v)
    assert_close(got, exp, "outside")
    assert not got[1].any()


def test_plan_longer_than_the_lengths(dev):
    """Splits of a plan made for 4000 keys over sequences of 31 to 700: the
    device's cut is finer than the plan's."""
    rng = np.random.default_rng(79)
    seq = [150, 700, 31]
    cfg, pt, ck0, cv0, q, _ = _case(rng, 16, seq, 0, 16)
    exp = oracle.decode_attention(q, ck0, cv0, pt, seq, cfg, 0, 0.05)
    got = _run_decode(dev, cfg, q, to_dev(ck0, dev), to_dev(cv0, dev), pt, seq, 0, 0.05, 200, 20)
    assert_close(got, exp, "finer cut")


def test_step_plans_by_capacity(dev):
    """A step's global layer over a cache far larger than its sequence (20480
    slots, 1100 keys): cut by the length for a single sequence too."""
    import torch
    rng = np.random.default_rng(80)
    n, page, pages = 1100, 64, 320
    cfg = cache_config(1, 1, page, pages, 1, 512, 0)
    pt = fill_page_table(cfg, [n])
    ck0 = np.full((pages * page, 1, 512), NAN)
    cv0 = ck0.copy()
    ck0[:n], cv0[:n] = randn_bf16(rng, (n, 1, 512)), randn_bf16(rng, (n, 1, 512))
    q, k, v = (randn_bf16(rng, (1, h, 512)) for h in (16, 1, 1))
    exp_k, exp_v = ck0.copy(), cv0.copy()
    oracle.kv_cache_write(exp_k, exp_v, cfg, pt, [0], [n - 1], 0, k, v)
    exp = oracle.decode_attention(q, exp_k, exp_v, pt, [n], cfg, 0, 0.0442)
    c = gk.make_config(*cfg)
    ws = torch.empty(gk.decode_step_workspace_bytes(1) // 4, dtype=torch.int32, device=dev)
    gk.check(gk.decode_step_workspace_init(ws, 1))
    ck, cv, out = to_dev(ck0, dev), to_dev(cv0, dev), to_dev(np.zeros_like(q), dev)
    seq, pos = to_dev(np.int32([n]), dev), to_dev(np.int32([n - 1]), dev)
    gk.check(gk.decode_step_layers_bf16(out, to_dev(q, dev), to_dev(k, dev), to_dev(v, dev), None, None, None, c,
                                        ck, cv, to_dev(pt, dev), c, seq, pos, 5, 1, 0.0442, 1, ws))
    torch.cuda.synchronize()
    assert gk.decode_step_status(ws) == 0
    assert np.array_equal(from_dev_bf16(ck).reshape(exp_k.shape), exp_k)
    assert_close(from_dev_bf16(out), exp, "capacity plan")


@pytest.mark.parametrize("split,seq", [
    (64, [300]),               # one-step splits, four waves
    (160, [450]),              # several steps, two waves
    (512, [200]),              # a single split
    (200, [150, 700, 31]),     # cut by the lengths
])
def test_infinite_values(dev, split, seq):
    """An infinite V element of one live key makes its dim infinite, with its
    sign, in every head; all others stay finite and right."""
    rng = np.random.default_rng(split + 7)
    cfg, pt, ck, cv, q, splits = _case(rng, split, seq, 0, 16)
    max_pages = cfg[3]
    for b, n in enumerate(seq):
        for key, dim, bits in ((n // 2, 5, 0x7F80), (n - 1, 200, 0xFF80), (0, 511, 0x7F80)):
            cv[pt[b * max_pages + key // 16] * 16 + key % 16, 0, dim] = bits
    exp = oracle.decode_attention(q, ck, cv, pt, seq, cfg, 0, 0.0442)
    got = _run_decode(dev, cfg, q, to_dev(ck, dev), to_dev(cv, dev), pt, seq, 0, 0.0442, split, splits)
    infinite = (exp & 0x7FFF) == 0x7F80
    assert infinite.sum() == 3 * 16 * len(seq)
    assert np.array_equal(got[infinite], exp[infinite])
    assert_close(np.where(infinite, 0, got), np.where(infinite, 0, exp), "finite dims")


def test_keys_past_the_plan_are_not_attended_to(dev):
    """A plan of fewer keys than a sequence holds covers the first split_size *
    num_splits of them, in a batch cut by its lengths as in a single sequence."""
    rng = np.random.default_rng(81)
    seq, split, splits = [700, 150, 310], 70, 3
    cfg, pt, ck, cv, q, _ = _case(rng, split, seq, 0, 16)
    covered = [min(n, split * splits) for n in seq]
    exp = oracle.decode_attention(q, ck, cv, pt, covered, cfg, 0, 0.0442)
    got = _run_decode(dev, cfg, q, to_dev(ck, dev), to_dev(cv, dev), pt, seq, 0, 0.0442, split, splits)
    assert_close(got, exp, "batch")
    one = cache_config(1, 1, 16, cfg[3], 1, 512, 0)
    got = _run_decode(dev, one, q[:1], to_dev(ck, dev), to_dev(cv, dev), pt[:cfg[3]], seq[:1], 0, 0.0442, split,
                      splits)
    assert_close(got, exp[:1], "single")


# (split size, keys held, live lengths, token positions, split counters)
RAW_CASES = [
    (65, [66], [66], [65], False),                      # two waves: a step and one key
    (96, [300], [300], [299], False),
    (160, [700], [700], [699], False),                  # the second page lookup
    (512, [512], [512], [511], False),                  # a single split, written directly
    (16, [4001, 17, 2900], [4001, 17, 2900], [4000, 16, 2899], False),  # cut by the lengths
    (96, [700, 40, 16, 333], [700, 20, 0, 333], [699, 33, 4, -1], False),  # tokens outside the live keys, none
    (64, [300, 65], [300, 65], [299, 64], True),
    (160, [700, 90], [700, 90], [699, 89], True),       # counters: four waves, several steps
    (333, [1000, 40, 333], [1000, 20, 333], [999, 33, -1], True),
]


@pytest.mark.parametrize("split,held,seq,pos,counters", RAW_CASES)
def test_raw_projections(dev, split, held, seq, pos, counters):
    """The fused preparation (q, the token's K and its V from the raw K) in
    both workgroup forms, cut by the lengths or not, combined by a launch or by
    the counters: outputs and cache rows each on their own."""
    import torch
    rng = np.random.default_rng(split * 31 + len(seq))
    cfg, pt, ck0, cv0, q, splits = _case(rng, split, held, 0, 16)
    print(f"raw split {split}x{splits} seq {seq} pos {pos} counters {counters}", flush=True)
    batch, max_pages, half = len(seq), cfg[3], 64
    k = randn_bf16(rng, (batch, 1, 512), scale=3.0)
    qw, kw = (oracle.f32_to_bf16(1.0 + 0.2 * rng.standard_normal(512).astype(np.float32)) for _ in range(2))
    cos, sin = oracle.fill_rope_tables(max(held), half, 1_000_000.0, 512)
    exp_k, exp_v, q_used, changed = ck0.copy(), cv0.copy(), q.copy(), []
    for b, p in enumerate(pos):
        if p < 0:
            continue
        c_row, s_row = cos[p * half:(p + 1) * half], sin[p * half:(p + 1) * half]
        for h in range(16):
            q_used[b, h] = oracle.prep_head(q[b, h], qw, c_row, s_row, 128)
        row = pt[b * max_pages + p // 16] * 16 + p % 16
        exp_k[row, 0] = oracle.prep_head(k[b, 0], kw, c_row, s_row, 128)
        exp_v[row, 0] = oracle.prep_head(k[b, 0], None, None, None, 128)
        changed.append(row)
    exp = oracle.decode_attention(q_used, exp_k, exp_v, pt, seq, cfg, 0, 0.0442)

    n = batch * 16 * splits
    pm, pl, pa = (torch.full((n * d,), float("nan"), device=dev) for d in (1, 1, 512))
    cnt = torch.zeros(batch, dtype=torch.int32, device=dev) if counters else None
    ck, cv, out = to_dev(ck0, dev), to_dev(cv0, dev), to_dev(np.full_like(q, NAN), dev)
    gk.check(gk.flash_attention_prep_append_decode_paged_bf16(
        out, pm, pl, pa, to_dev(q, dev), ck, cv, to_dev(pt, dev), to_dev(np.int32(seq), dev),
        to_dev(np.int32(pos), dev), to_dev(k, dev), None, to_dev(qw, dev), to_dev(kw, dev), to_dev(cos, dev),
        to_dev(sin, dev), gk.make_config(*cfg), 0, 0.0442, split, splits, batch, split_counters=cnt))
    torch.cuda.synchronize()
    assert not counters or not cnt.any().item()
    got_k, got_v = (from_dev_bf16(x).reshape(ck0.shape) for x in (ck, cv))
    rest = np.setdiff1d(np.arange(len(ck0)), changed)
    assert np.array_equal(got_k[rest], ck0[rest]) and np.array_equal(got_v[rest], cv0[rest])
    _close_bits(got_k[changed], exp_k[changed], "cache K")
    _close_bits(got_v[changed], exp_v[changed], "cache V")
    assert_close(from_dev_bf16(out).reshape(exp.shape), exp, "attention")
