"""Selection of at most 64 keys, by one wavefront's registers and, where they or
its candidates do not hold it, by all wavefronts of a workgroup, in the
selection op and in the fused step: the oracle's indices and order exactly.
Keys are the first component of each summary row (q is its unit vector), so
scores carry no rounding."""
import numpy as np
import pytest
import torch

import oracle
from csahca_amd import native

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _summary(values, D):
    s = torch.zeros(*values.shape, D)
    s[..., 0] = values
    return s


def _values(kind, bh, C):
    g = torch.Generator().manual_seed(C + bh)
    v = torch.randn(1, bh, C, generator=g)
    if kind == "ties":                   # four values: more keys at the threshold than candidates
        v = torch.randint(0, 4, (1, bh, C), generator=g).float()
    elif kind == "rising":               # the top keys lie side by side at the end
        v = v.sort(dim=-1).values
    elif kind == "strided":              # the top keys 256 apart, in one column of the walk but for its rotation
        v[..., ::256] += 100.0
    elif kind == "negative infinity":
        v[..., 3:] = float("-inf")
    return v


@pytest.mark.parametrize("kind", ["random", "ties", "rising", "strided", "negative infinity"])
@pytest.mark.parametrize("C,k", [(64, 64), (65, 40), (65, 41), (128, 40), (129, 33), (255, 33), (257, 64), (512, 41),
                                 (2048, 33), (2049, 1), (2303, 64), (2305, 8), (4096, 64), (6295, 14), (14003, 63), (20001, 64),
                                 (2500, 65), (129, 1), (192, 36), (192, 37), (256, 36), (512, 34)])
def test_selection_and_step_match_the_oracle(kind, C, k):
    H, D, chunk = 3, 64, 2
    summ = _summary(_values(kind, H, C), D)
    q = torch.zeros(1, H, D)
    q[..., 0] = 1.0
    q = q.to(torch.bfloat16)
    want, _ = oracle.select_topk(q, summ, k)
    qd, sd = q.to(DEV), summ.to(DEV)
    got = native.csa_select_topk(qd, sd, k)
    assert np.array_equal(got.cpu().numpy(), want)
    g = torch.Generator().manual_seed(7)
    kc, vc = (torch.randn(1, H, C * chunk, D, generator=g).to(torch.bfloat16) for _ in range(2))
    out, idx = native.csa_decode_step(qd, kc.to(DEV), vc.to(DEV), sd, chunk, k)
    assert np.array_equal(idx.cpu().numpy(), want)
    ref = oracle.csa_attend(q, kc, vc, torch.from_numpy(np.asarray(want)), chunk, prob_dtype=oracle.F32)
    diff = np.abs(out.double().cpu().numpy() - ref)
    assert np.all(diff <= 2e-2 + 1e-2 * np.abs(ref)), f"max_abs={diff.max():.3e}"


@pytest.mark.parametrize("count", [3, 200, 256, 257, 2049])
def test_step_with_a_device_count(count):
    """A capacity of more than 2048 chunks, few of them in play."""
    H, D, chunk, C, k = 2, 64, 2, 3000, 16
    summ = _summary(_values("random", H, C), D)
    q = torch.zeros(1, H, D)
    q[..., 0] = 1.0
    q = q.to(torch.bfloat16)
    g = torch.Generator().manual_seed(9)
    kc, vc = (torch.randn(1, H, C * chunk, D, generator=g).to(torch.bfloat16) for _ in range(2))
    n = torch.tensor([count], dtype=torch.int32, device=DEV)
    _, idx = native.csa_decode_step_dev(q.to(DEV), kc.to(DEV), vc.to(DEV), summ.to(DEV), n, chunk, k)
    want, _ = oracle.select_topk(q, summ[:, :, :count], min(k, count))
    full = np.full((1, H, k), -1, dtype=np.int64)
    full[..., :min(k, count)] = want
    assert np.array_equal(idx.cpu().numpy(), full)


@pytest.mark.parametrize("kind", ["random", "ties", "rising", "strided"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("C,k", [(1, 1), (63, 32), (64, 8), (127, 9), (128, 40), (129, 8), (512, 32), (513, 8),
                                 (1023, 32), (1024, 9), (1025, 8)])
def test_register_sizes_of_the_step(kind, dtype, C, k):
    """head_dim 128 in 16 bits: at the edges of 2, 8, 16 and 32 keys per lane,
    by the host's count, by the device's, and beside the HCA pass."""
    H, D, chunk = 2, 128, 2
    summ = _summary(_values(kind, H, C), D)
    q = torch.zeros(1, H, D)
    q[..., 0] = 1.0
    q = q.to(dtype)
    want, _ = oracle.select_topk(q, summ, k)
    g = torch.Generator(device=DEV).manual_seed(C)
    kc, vc = (torch.randn(1, H, C * chunk, D, generator=g, device=DEV).to(dtype) for _ in range(2))
    qd, sd = q.to(DEV), summ.to(DEV)
    out, idx = native.csa_decode_step(qd, kc, vc, sd, chunk, k)
    assert np.array_equal(idx.cpu().numpy(), want)
    n = torch.tensor([C], dtype=torch.int32, device=DEV)
    _, idx = native.csa_decode_step_dev(qd, kc, vc, sd, n, chunk, k)
    assert np.array_equal(idx.cpu().numpy(), want)
    hyb = native.hybrid_decode_forward(qd, kc, vc, csa_chunk_size=chunk, csa_top_k=k, hca_chunk_size=chunk,
                                       csa_weight=1.0, summary=sd)
    diff = np.abs(hyb.double().cpu().numpy() - out.double().cpu().numpy())
    assert np.all(diff <= 2e-2 + 1e-2 * np.abs(out.double().cpu().numpy()))
