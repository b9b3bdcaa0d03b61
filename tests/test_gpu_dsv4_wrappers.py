"""The DSV4 wrappers convert what is not yet contiguous and of its type and
pass the rest on: the same bits either way, and for an absent tensor the same
as for an empty one."""
import pytest
import torch

from csahca_amd import extension
from csahca_amd.synthetic import make_dsv4_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _strided(t, dtype):
    """t's values in dtype, every other element of a larger tensor."""
    big = torch.zeros(*t.shape, 2, dtype=dtype, device=t.device)
    big[..., 0] = t.to(dtype)
    return big[..., 0]


@pytest.mark.parametrize("tiled", ["0", "1"])
@pytest.mark.parametrize("ratio", [0, 4])
def test_converted_and_absent_inputs(tiled, ratio, monkeypatch):
    monkeypatch.setenv("CSAHCA_DSV4_TILED", tiled)
    c = make_dsv4_case(compress_ratio=ratio, num_queries=3, heads=8, num_tokens=256, top_k=32, page_size=64,
                       extra_tokens=256, extra_top_k=16, seed=8, device=DEV)

    def call(q, cache, idx, lens, extra, sink):
        if ratio:
            return extension.dsv4_sparse_decode_forward(q, cache, idx, lens, *extra, sink, c.page_size,
                                                        c.extra_page_size, 0.05)
        return extension.dsv4_swa_decode_forward(q, cache, idx, lens, sink, c.page_size, 0.05)

    extra = (c.extra_cache, c.extra_token_indices, c.extra_topk_lengths) if ratio else None
    want = call(c.q, c.cache, c.token_indices, c.topk_lengths, extra, c.attn_sink)
    other = (c.extra_cache.view(torch.float8_e4m3fn), _strided(c.extra_token_indices, torch.int64),
             _strided(c.extra_topk_lengths, torch.int64)) if ratio else None
    got = call(_strided(c.q, c.q.dtype), c.cache.view(torch.float8_e4m3fn), _strided(c.token_indices, torch.int64),
               _strided(c.topk_lengths, torch.int64), other, _strided(c.attn_sink, torch.float64))
    assert torch.equal(got, want)
    none = lambda dtype: torch.empty(0, dtype=dtype, device=DEV)
    absent = call(c.q, c.cache, c.token_indices, None, extra and (*extra[:2], None), None)
    empty = call(c.q, c.cache, c.token_indices, none(torch.int32), extra and (*extra[:2], none(torch.int32)),
                 none(torch.float32))
    assert torch.equal(absent, empty)
