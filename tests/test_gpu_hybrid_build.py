"""The hybrid op that builds its own chunk summaries, over the shapes at which
it reads K once and beside them: the bits of the summary kernel, the decode
step and the blended HCA op in turn."""
import pytest
import torch

from csahca_amd import native

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, F16, F32, F64 = torch.bfloat16, torch.float16, torch.float32, torch.float64


@pytest.mark.parametrize("B,H,S,D,dtype,chunk,hca", [
    (2, 8, 32768, 128, BF, 64, 256),
    (1, 8, 8192, 128, BF, 64, 64),       # one summary chunk to an HCA chunk
    (1, 3, 6400, 128, F16, 64, 128),     # 150 items; the last batch of rows of a wavefront full
    (1, 1, 48 * 73 * 3, 128, BF, 48, 144),   # an odd count of items, batches that end inside a chunk
    (3, 2, 16 * 300, 128, F16, 16, 16),  # one step of row groups per chunk
    (2, 4, 112 * 20, 128, BF, 112, 448),
    (1, 8, 8192, 64, BF, 64, 256),       # 8 rows a load
    (1, 5, 4096, 64, F16, 32, 32),
    (1, 8, 8192, 256, F16, 64, 128),     # 2 rows a load
    (1, 2, 8 * 600, 256, BF, 8, 24),
    (1, 4, 4096, 64, F32, 64, 128),
    (2, 8, 8192, 128, F32, 64, 256),
    (1, 3, 100 * 24, 256, F32, 100, 400),
    (1, 2, 6400, 128, BF, 100, 400),     # no whole row groups: two reads
    (1, 2, 6144, 128, BF, 64, 96),       # an HCA chunk of one and a half: two reads
    (1, 2, 6144, 128, BF, 128, 64),      # smaller HCA chunks: two reads
    (1, 2, 4096, 96, BF, 64, 256),       # head_dim 96: two reads
    (1, 2, 4096, 128, F64, 64, 256),     # fp64: two reads
])
@pytest.mark.parametrize("one_read", [None, "1"])
def test_equals_the_ops_in_turn(B, H, S, D, dtype, chunk, hca, one_read, monkeypatch):
    if one_read is not None:  # wherever the shape allows it, whatever the size
        monkeypatch.setenv("CSAHCA_HYBRID_ONE_READ", one_read)
    g = torch.Generator(device=DEV).manual_seed(S + D + chunk)
    q = torch.randn(B, H, D, generator=g, device=DEV).to(dtype)
    k, v = (torch.randn(B, H, S, D, generator=g, device=DEV).to(dtype) for _ in range(2))
    summ = native.csa_chunk_summary(k, chunk)
    csa, _ = native.csa_decode_step(q, k, v, summ, chunk, 5)
    want = native.hca_decode_forward(q, k, v, hca, blend=csa, csa_weight=0.7)
    got = native.hybrid_decode_forward(q, k, v, csa_chunk_size=chunk, csa_top_k=5, hca_chunk_size=hca)
    assert torch.equal(got, want)
    assert all(x == 0 for x in native.csa_step_status().values())


def test_unaligned_caches(monkeypatch):
    """K and V 8 bytes past a 16-byte boundary: two reads, by the generic kernels."""
    monkeypatch.setenv("CSAHCA_HYBRID_ONE_READ", "1")
    g = torch.Generator(device=DEV).manual_seed(3)
    q = torch.randn(1, 2, 128, generator=g, device=DEV).to(BF)
    k, v = (torch.randn(4 + 2 * 2048 * 128, generator=g, device=DEV).to(BF)[4:].view(1, 2, 2048, 128)
            for _ in range(2))
    assert k.data_ptr() % 16 == 8
    want = native.hca_decode_forward(q, k, v, 256, blend=native.csa_decode_step(
        q, k, v, native.csa_chunk_summary(k, 64), 64, 4)[0], csa_weight=0.7)
    assert torch.equal(native.hybrid_decode_forward(q, k, v, csa_chunk_size=64, csa_top_k=4, hca_chunk_size=256), want)


def test_graph_replays(monkeypatch):
    """Captured, replayed with eager work between the replays."""
    monkeypatch.setenv("CSAHCA_HYBRID_ONE_READ", "1")
    g = torch.Generator(device=DEV).manual_seed(5)
    q = torch.randn(1, 8, 128, generator=g, device=DEV).to(BF)
    k, v = (torch.randn(1, 8, 8192, 128, generator=g, device=DEV).to(BF) for _ in range(2))
    run = lambda: native.hybrid_decode_forward(q, k, v, csa_chunk_size=64, csa_top_k=8, hca_chunk_size=256)
    want = run()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = run()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(run(), want)
