"""Chunk-causal grids of more than one round of CUs deal their q-tiles longest first over all heads;
every (head, q-tile) must still be computed exactly once.  Heads that are a multiple of 8, of 4 and
odd, two streams, ragged last q-tiles and 4-wave groups, against float64 masked attention on the GPU
(bars of tests/helpers.py)."""

import pytest
import torch

from solarwm_amd import chunk_causal_attention

from .helpers import assert_attn_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,L,chunk,dtype", [
    (1, 40, 1700, 150, torch.bfloat16),   # 7 q-tiles x 40 heads
    (2, 6, 6000, 777, torch.bfloat16),    # 24 x 12, chunk limits inside tiles
    (1, 37, 1801, 64, torch.float32),     # odd head count
    (3, 43, 400, 100, torch.bfloat16),    # 2 q-tiles x 129: the second round holds one workgroup
    (1, 300, 320, 80, torch.bfloat16),    # as many heads as CUs, 4-wave groups: the plain order
    (2, 150, 450, 60, torch.bfloat16),    # the same with 8-wave groups: longest first
])
def test_longest_first_chunk_causal(gpu, B, H, L, chunk, dtype):
    print("causal order", B, H, L, chunk, dtype, flush=True)
    g = torch.Generator(device=gpu).manual_seed(L)
    q, k, v = (torch.randn(B, L, H, 128, generator=g, device=gpu).to(dtype) for _ in range(3))
    got = chunk_causal_attention(q, k, v, chunk_tokens=chunk)
    pos = torch.arange(L, device=gpu)
    hidden = pos[None, :] >= ((pos // chunk + 1) * chunk)[:, None]
    want = torch.empty(B, L, H, 128, dtype=torch.float64)
    for b in range(B):
        for h in range(H):
            # the kernels round float32 inputs to bf16
            qh, kh, vh = (x[b, :, h].to(torch.bfloat16).double().contiguous() for x in (q, k, v))
            s = (qh @ kh.t().contiguous()) * 128 ** -0.5
            want[b, :, h] = (s.masked_fill(hidden, float("-inf")).softmax(-1) @ vh).cpu()
    assert_attn_close(got, want)
