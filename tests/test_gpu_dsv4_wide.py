"""The DSV4 kernel for many heads and queries (64 heads and the whole slot list
in one workgroup) against the CPU oracle, at the edges of its tiles: 16-slot
sub-tiles, 64-slot rounds, 64-head groups, odd pages.  CSAHCA_DSV4_WIDE=1 routes
these small calls to it.  Tolerance: the FP8-cache bar |got - ref| <= 5e-2 +
5e-2 |ref|, unless a test says otherwise."""
import math

import numpy as np
import pytest
import torch

import oracle
from csahca_amd import extension, native
from csahca_amd.dsv4_layout import pack_dsv4_cache
from csahca_amd.synthetic import make_dsv4_case

pytestmark = pytest.mark.gpu
DEV = "cuda"
SCALE = 1.0 / math.sqrt(512)


@pytest.fixture(autouse=True)
def _wide(monkeypatch):
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    native.lib()
    monkeypatch.setenv("CSAHCA_DSV4_WIDE", "1")


def gpu_out(c, sink=True):
    d = lambda t: None if t is None else t.to(DEV)
    s = d(c.attn_sink) if sink else None
    if c.extra_cache is not None:
        return extension.dsv4_sparse_decode_forward(d(c.q), d(c.cache), d(c.token_indices), d(c.topk_lengths),
                                                    d(c.extra_cache), d(c.extra_token_indices),
                                                    d(c.extra_topk_lengths), s, c.page_size, c.extra_page_size, SCALE)
    return extension.dsv4_swa_decode_forward(d(c.q), d(c.cache), d(c.token_indices), d(c.topk_lengths), s,
                                             c.page_size, SCALE)


def oracle_out(c, sink=True):
    kw = {}
    if c.extra_cache is not None:
        kw = dict(extra_cache=c.extra_cache.cpu(), extra_token_indices=c.extra_token_indices.cpu(),
                  extra_topk_lengths=None if c.extra_topk_lengths is None else c.extra_topk_lengths.cpu(),
                  extra_page_size=c.extra_page_size)
    return oracle.dsv4_reference_attention(c.q.cpu(), c.cache.cpu(), c.token_indices.cpu(),
                                           None if c.topk_lengths is None else c.topk_lengths.cpu(),
                                           c.attn_sink.cpu() if sink else None, page_size=c.page_size,
                                           softmax_scale=SCALE, **kw)


def assert_close(got, ref, atol=5e-2, rtol=5e-2):
    g = got.detach().double().cpu().numpy()
    assert g.shape == ref.shape
    assert np.array_equal(np.isnan(g), np.isnan(ref))
    diff = np.abs(np.nan_to_num(g) - np.nan_to_num(ref))
    bad = diff > atol + rtol * np.abs(np.nan_to_num(ref))
    assert not bad.any(), f"max_abs={diff.max():.3e} bad={int(bad.sum())}/{bad.size}"


def assert_norm(got, ref):
    """Each query's relative norm (over its heads and dims) within 2^-8: the
    output's rounding to bf16, at most 2^-9 of each value, and that of the
    weights, at most 2^-9 of each and independent over rows of independent
    directions, hence at most 2^-9 of the output's norm."""
    g = got.detach().double().cpu().numpy()
    err = np.linalg.norm(g - ref, axis=(1, 2))
    norm = np.linalg.norm(ref, axis=(1, 2))
    assert (err <= 2.0**-8 * norm).all(), err / norm


@pytest.mark.parametrize("heads,top_k,extra_top_k,page,extra_page", [
    (64, 1, 0, 64, 0),        # one slot
    (17, 15, 0, 64, 0),       # less than a sub-tile; 17 of 64 heads
    (64, 16, 1, 64, 16),      # a full sub-tile and one slot of the other list
    (33, 17, 15, 48, 48),     # pages that are no power of two
    (64, 63, 0, 1, 0),        # pages of one token
    (65, 64, 64, 64, 16),     # whole rounds; a second head group of one head
    (70, 65, 33, 64, 100),    # one slot into a round
    (64, 128, 64, 256, 64),   # the window and its C4 entries
    (24, 128, 512, 64, 1),    # ten rounds
    (128, 100, 157, 64, 64),  # ragged in both lists
])
@pytest.mark.parametrize("lengths", ["full", "ragged", "none"])
def test_wide_kernel_matches_oracle(heads, top_k, extra_top_k, page, extra_page, lengths):
    c = make_dsv4_case(compress_ratio=4 if extra_top_k else 0, num_queries=9, heads=heads, num_tokens=700, top_k=top_k,
                       page_size=page, extra_tokens=600, extra_top_k=extra_top_k, extra_page_size=extra_page or None,
                       full_lengths=lengths == "full", seed=heads + top_k, device="cpu")
    if lengths == "ragged":
        c.topk_lengths[0] = 0                     # no window slots: the second list starts the first round
        c.topk_lengths[1] = min(top_k, 5)
        c.token_indices[2, 0] = -1
        c.token_indices[3, :] = -1                # a whole list of skipped slots
        if extra_top_k:
            c.extra_topk_lengths[1] = 0
            c.extra_topk_lengths[4] = 1
            c.extra_token_indices[5, 0] = 10_000_000  # a page past the cache
    elif lengths == "none":
        c.topk_lengths = None
        c.extra_topk_lengths = None
    for sink in (True, False):
        got, ref = gpu_out(c, sink), oracle_out(c, sink)
        assert_close(got, ref)
        assert_norm(got, ref)


def excess_bits(c, rows):
    """Per query, how far (log2) the best later score of any head exceeds that
    head's maximum over the first 64 slots."""
    x = torch.einsum("qhd,sd->qhs", c.q.double(), rows.to(torch.bfloat16).double()) * SCALE / math.log(2)
    return (x[..., 64:].amax(-1) - x[..., :64].amax(-1)).amax(-1)


@pytest.mark.parametrize("jump,low,high", [
    (0.5, -math.inf, 7), (2.0, 9, 60), (4.0, 18, 60), (8.0, 36, 62), (40.0, 80, math.inf), (4000.0, 80, math.inf),
])
def test_wide_kernel_scores_that_outgrow_the_first_round(jump, low, high):
    """Probabilities are formed against the first round's maximum: later scores
    that exceed it by up to 2^8 and by up to 2^64 are kept as they are, larger
    ones take the second walk.  `low` and `high` bound the excess of every
    query, with room for the cache's rounding of the rows, so that each stays
    in its regime.  Against the oracle."""
    c = make_dsv4_case(compress_ratio=0, num_queries=5, heads=64, num_tokens=512, top_k=200, page_size=64,
                       full_lengths=True, seed=3, pack=False, device="cpu")
    c.token_indices = torch.arange(200, dtype=torch.int32).repeat(5, 1)
    rows = c.k_tokens.float()
    rows[:64] *= 0.01
    rows[130:] *= jump
    excess = excess_bits(c, rows[:200])
    assert low < excess.min() and excess.max() < high, excess
    c.cache = pack_dsv4_cache(rows.to(torch.bfloat16), page_size=64)
    ref = oracle_out(c)
    # the outputs are of the rows' own magnitude: the bar relative to it
    assert_close(gpu_out(c) / max(jump, 1.0), ref / max(jump, 1.0))


def test_wide_kernel_accumulators_that_overflow_the_first_walk():
    """A late score 40 bits above the first round's maximum over rows of 1e28: the
    accumulators overflow against that maximum, not against the true one, so
    the list is walked again."""
    c = make_dsv4_case(compress_ratio=0, num_queries=3, heads=64, num_tokens=200, top_k=200, page_size=64,
                       full_lengths=True, seed=5, pack=False, device="cpu")
    c.token_indices = torch.arange(200, dtype=torch.int32).repeat(3, 1)
    c.q[:, :, 500], c.q[:, :, 510] = 8.0, 0.0
    c.k_tokens[:, 500], c.k_tokens[:, 510] = 0.0, 1e28
    c.k_tokens[150, 500] = 40 * math.log(2) * math.sqrt(512) / 8.0
    excess = excess_bits(c, c.k_tokens)
    assert 28 < excess.min() and excess.max() < 60, excess
    c.cache = pack_dsv4_cache(c.k_tokens, page_size=64)
    ref = oracle_out(c)
    assert np.isfinite(ref).all() and abs(ref[..., 510]).min() > 5e27
    assert_close(gpu_out(c), ref)


def test_wide_kernel_scale_byte_255_poisons_its_query_only():
    c = make_dsv4_case(compress_ratio=0, num_queries=4, heads=64, num_tokens=256, top_k=70, page_size=64,
                       full_lengths=True, seed=8, device="cpu")
    c.token_indices = (torch.arange(70, dtype=torch.int32)[None] + 64 * torch.arange(4, dtype=torch.int32)[:, None]) % 250
    c.token_indices[:, :] = torch.where(c.token_indices == 200, 0, c.token_indices)
    c.token_indices[2, 67] = 200  # only query 2 sees row 200
    sb = 64 * 576 + (200 % 64) * 8
    c.cache[200 // 64, sb + 3] = 255
    ref = oracle_out(c)
    assert np.isnan(ref[2]).all() and np.isfinite(ref[[0, 1, 3]]).all()
    assert_close(gpu_out(c), ref)


def test_wide_kernel_decodes_every_code_exactly():
    """One valid slot and no sink: the output is the dequantised row, for every
    finite e4m3 code under scale bytes over their range."""
    scales = [0, 1, 90, 120, 127, 140, 200, 246]
    cache = torch.zeros(8, 64 * 584 // 576 * 576 + 576, dtype=torch.uint8)
    codes = torch.tensor([b for b in range(256) if b & 0x7F != 0x7F], dtype=torch.uint8)
    for i, s in enumerate(scales):
        cache[i, :448] = codes.roll(7 * i).repeat(2)[:448]
        cache[i, 64 * 576:64 * 576 + 7] = s
    q = torch.randn(8, 64, 512, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16) * 1e-30
    out = extension.dsv4_swa_decode_forward(q.to(DEV), cache.to(DEV),
                                            (64 * torch.arange(8, dtype=torch.int32))[:, None].to(DEV), None, None, 64,
                                            SCALE)
    want = oracle.dsv4_reference_attention(q, cache, (64 * torch.arange(8, dtype=torch.int32))[:, None], None, None,
                                           page_size=64, softmax_scale=SCALE)
    got = out.double().cpu().numpy()
    assert np.array_equal(got, torch.from_numpy(np.asarray(want)).to(torch.bfloat16).double().numpy())


def relative_error(got, ref):
    return np.linalg.norm(got.double().cpu().numpy() - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("q_scale,nats", [(1.0, 0.0), (2.0, 0.0), (4.0, 0.0), (1.0, 4.0), (1.0, 8.0), (1.0, 12.0),
                                          (1.0, 20.0)])
def test_wide_kernel_is_as_exact_as_the_kernel_it_stands_in_for(monkeypatch, q_scale, nats):
    """Error against 64 bits (relative norm over 131072 values) of flat and of
    peaked scores: one key past the first round `nats` above the rest weighs
    nearly everything.  Not above the per-query kernel's, whose maximum moves:
    3% for the spread of two independent sets of roundings, 1e-5 where both
    outputs are nearly the key itself."""
    c = make_dsv4_case(compress_ratio=0, num_queries=4, heads=64, num_tokens=640, top_k=640, page_size=64,
                       full_lengths=True, seed=11, pack=False, device="cpu")
    c.token_indices = torch.arange(640, dtype=torch.int32).repeat(4, 1)
    c.q = (c.q.float() * q_scale).to(torch.bfloat16)
    if nats:
        c.q[:, :, 500] = 8.0  # a bf16 dim of the latent that only row 300 has
        c.k_tokens[:, 500] = 0.0
        c.k_tokens[300, 500] = nats * math.sqrt(512) / 8.0
    c.cache = pack_dsv4_cache(c.k_tokens, page_size=64)
    ref = oracle_out(c)
    wide = relative_error(gpu_out(c), ref)
    monkeypatch.setenv("CSAHCA_DSV4_WIDE", "0")
    monkeypatch.setenv("CSAHCA_DSV4_QUERY", "1")
    other = relative_error(gpu_out(c), ref)
    print(f"q x {q_scale}, {nats} nats: wide {wide:.6f}, per-query {other:.6f}")
    assert wide <= 1.03 * other + 1e-5


def call_us(calls):
    """Time of one call in us for each of `calls`, taken in turn: the least of
    nine graph replays of eight calls."""
    graphs = []
    for call in calls:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            for _ in range(8):
                call()
        graphs.append(graph)
    us = [math.inf] * len(calls)
    for _ in range(10):  # (the first replay of each warms up)
        for i, graph in enumerate(graphs):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            us[i] = min(us[i], start.elapsed_time(end) * 1e3 / 8)
    return us


def swa_call(c, cache, indices):
    args = (c.q.to(DEV), cache.to(DEV), indices.to(DEV), c.topk_lengths.to(DEV), c.attn_sink.to(DEV))
    return lambda: extension.dsv4_swa_decode_forward(*args, c.page_size, SCALE)


def test_wide_kernel_pad_byte_is_not_a_scale():
    """The eighth scale byte of a token holds whatever the cache's memory did:
    0xFF there neither changes the output nor sends the tiles through the
    general decode (1.3 times the time)."""
    c = make_dsv4_case(compress_ratio=0, num_queries=64, heads=64, num_tokens=4096, top_k=640, page_size=64,
                       full_lengths=True, seed=13, device="cpu")
    padded = c.cache.clone()
    for slot in range(64):
        padded[:, 64 * 576 + 8 * slot + 7] = 255
    plain, pad = swa_call(c, c.cache, c.token_indices), swa_call(c, padded, c.token_indices)
    assert torch.equal(plain(), pad())
    t_plain, t_pad = call_us([plain, pad])
    assert t_pad < 1.12 * t_plain, f"{t_pad:.2f} us with pad bytes of 255, {t_plain:.2f} without"


@pytest.mark.parametrize("skipped", [64, 100, 192])
def test_wide_kernel_skipped_slots_first(skipped):
    """A list whose first rounds hold no row takes its maximum from the first
    round that does, in one walk: two take 1.8 times as long as the full list,
    one walk 1.03 to 1.13 times (the masks of a round of skipped slots cost
    1.2 us)."""
    c = make_dsv4_case(compress_ratio=0, num_queries=64, heads=64, num_tokens=4096, top_k=640, page_size=64,
                       full_lengths=True, seed=17, device="cpu")
    indices = c.token_indices.clone()
    indices[:, :skipped] = -1
    full, late = swa_call(c, c.cache, c.token_indices), swa_call(c, c.cache, indices)
    t_full, t_late = call_us([full, late])
    c.q, c.token_indices, c.topk_lengths = c.q[:4], indices[:4], c.topk_lengths[:4]
    assert_close(late()[:4], oracle_out(c))
    assert t_late < 1.3 * t_full, f"{t_late:.2f} us with {skipped} slots skipped, {t_full:.2f} without"


def kernels_of(call):
    with native.profile_launches() as p:
        call()
        torch.cuda.synchronize()
    return set(p.results)


@pytest.mark.parametrize("nq,heads,slots,wide", [
    (72, 64, 257, True),    # more (query, 16 heads) pairs than CUs
    (72, 64, 256, False),   # the longest list of the one-pass kernel
    (64, 64, 384, False),   # 256 pairs
    (64, 64, 447, False),
    (64, 64, 448, True),
    (33, 64, 448, True),    # 132 pairs
    (32, 64, 448, False),   # 128 pairs
    (32, 64, 575, False),
    (32, 64, 576, True),
    (20, 64, 576, True),    # 80 pairs
    (19, 64, 576, False),
    (16, 64, 639, False),   # 64 pairs
    (16, 64, 640, True),
    (15, 64, 640, False),
    (1, 256, 384, False),   # 16 pairs, in a grid of 128
    (1, 256, 640, False),
    (4, 256, 640, True),    # 64 pairs
    (256, 16, 640, False),  # 16 heads: three quarters padding
])
def test_wide_kernel_takes_its_calls(monkeypatch, nq, heads, slots, wide):
    """The rule by itself, no switch set (on a device of 256 CUs)."""
    monkeypatch.delenv("CSAHCA_DSV4_WIDE")
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    c = make_dsv4_case(compress_ratio=0, num_queries=nq, heads=heads, num_tokens=700, top_k=slots, page_size=64,
                       seed=slots, device="cpu")
    call = swa_call(c, c.cache, c.token_indices)
    assert ("dsv4_wide_kernel" in kernels_of(call)) == wide
    out = call()[:2]
    c.q, c.token_indices, c.topk_lengths = c.q[:2], c.token_indices[:2], c.topk_lengths[:2]
    assert_close(out, oracle_out(c))
