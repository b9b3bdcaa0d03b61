"""The split-KV op where its split differs from the caller's tile, and the merge
of more than 64 partials per head, against the CPU oracle.  Tolerance: the bar
of this path, |got - ref| <= 2e-2 + 1e-2 |ref| for 16-bit storage, 1e-4 + 1e-4
|ref| for fp32 and fp64."""
import numpy as np
import pytest
import torch

import oracle
from csahca_amd import native

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,H,S,D,chunk,k,tile,dtype", [
    (1, 1, 8192, 128, 64, 128, 8, torch.bfloat16),     # 8192 slots: 64 tiles of 128, the last one-round-trip merge
    (1, 2, 12928, 128, 64, 202, 8, torch.bfloat16),    # 101 tiles
    (1, 1, 8256, 64, 64, 129, 1, torch.float16),       # 65 tiles: one past the one-round-trip merge
    (1, 1, 132000, 64, 1000, 132, 7, torch.float16),   # 1032 tiles: two passes of weights, 8 in the second
    (1, 1, 132000, 64, 1000, 132, 133, torch.float16), # 993 tiles of 133 slots, no whole load batches
    (1, 1, 140000, 64, 1000, 140, 8, torch.bfloat16),  # 1094 tiles: two passes of weights
    (2, 1, 9000, 96, 50, 180, 8, torch.bfloat16),      # generic kernel, 563 tiles; columns that are no multiple of 32
    (1, 2, 9216, 256, 48, 190, 3, torch.float32),      # 72 tiles of 128 slots
    (1, 1, 9216, 100, 64, 144, 8, torch.float64),      # generic kernel, 576 tiles, 100 columns
    (1, 3, 4352, 128, 64, 68, 64, torch.float32),      # 61 tiles of 72 slots for the asked 64
    (3, 2, 640, 128, 64, 3, 5, torch.bfloat16),        # 192 slots: tiles of 16 for the asked 5
    (1, 1, 64, 64, 16, 1, 3, torch.float16),           # 16 slots in one tile of at most 32
])
def test_split_matches_oracle(B, H, S, D, chunk, k, tile, dtype):
    g = torch.Generator().manual_seed(S + D + k)
    q = torch.randn(B, H, D, generator=g).to(dtype)
    kc = torch.randn(B, H, S, D, generator=g).to(dtype)
    vc = torch.randn(B, H, S, D, generator=g).to(dtype)
    C = S // chunk
    idx = torch.stack([torch.randperm(C, generator=g)[:k] for _ in range(B * H)]).view(B, H, k).to(torch.int32)
    idx[0, 0, 0] = -1                       # a skipped chunk
    if k > 100:
        idx[0, 0, 3:] = -1                  # most tiles of this head are empty
    ref = oracle.csa_attend(q, kc, vc, idx, chunk, prob_dtype=oracle.F32)
    got = native.csa_decode_forward_tiled(q.to(DEV), kc.to(DEV), vc.to(DEV), idx.to(DEV), chunk, tile)
    atol, rtol = (2e-2, 1e-2) if dtype in (torch.bfloat16, torch.float16) else (1e-4, 1e-4)
    diff = np.abs(got.double().cpu().numpy() - ref)
    assert np.all(diff <= atol + rtol * np.abs(ref)), f"max_abs={diff.max():.3e}"


def test_split_near_int32_slots():
    """2^31 - 16384 slots: the last of 8192 tiles of 262144 would end past int32.
    Only the last 8 chunks, all in that tile, hold an id."""
    chunk, k, S, D = 16384, 131071, 32768, 64
    g = torch.Generator().manual_seed(7)
    q = torch.randn(1, 1, D, generator=g).to(torch.bfloat16)
    kc = torch.randn(1, 1, S, D, generator=g).to(torch.bfloat16)
    vc = torch.randn(1, 1, S, D, generator=g).to(torch.bfloat16) + 1.0
    idx = torch.full((1, 1, k), -1, dtype=torch.int32)
    idx[..., -8:] = 1
    # (the same chunk 8 times: the softmax is that of the chunk once)
    ref = oracle.csa_attend(q, kc, vc, torch.ones(1, 1, 1, dtype=torch.int32), chunk, prob_dtype=oracle.F32)
    got = native.csa_decode_forward_tiled(q.to(DEV), kc.to(DEV), vc.to(DEV), idx.to(DEV), chunk, 128)
    diff = np.abs(got.double().cpu().numpy() - ref)
    assert np.all(diff <= 2e-2 + 1e-2 * np.abs(ref)), f"max_abs={diff.max():.3e}"
