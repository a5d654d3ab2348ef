"""How many vocabulary rows a backward stages together (``swvr_bwd_tiling``; no GPU needed): a power
of two of chunks up to what 8192 tokens would take at the caller's chunk, 256 MB of packed W at most,
and the chunk itself from 4097 tokens on or when it is below the default."""
import pytest
import torch

from swvr_amd import _lib


@pytest.mark.parametrize("dtype,N,K,V,chunk,C", [
    (torch.bfloat16, 500, 1024, 151936, 8192, 16 * 8192),
    (torch.bfloat16, 500, 1024, 32000, 8192, 32000),         # the whole vocabulary, in tiles of 256
    (torch.bfloat16, 1, 256, 10**6, 8192, 32 * 8192),        # 256 padded positions
    (torch.bfloat16, 500, 4096, 151936, 8192, 4 * 8192),     # 256 MB of packed W
    (torch.float32, 500, 4096, 151936, 8192, 2 * 8192),
    (torch.bfloat16, 2048, 1024, 151936, 8192, 4 * 8192),
    (torch.bfloat16, 2049, 1024, 151936, 8192, 2 * 8192),
    (torch.bfloat16, 4096, 1024, 151936, 8192, 2 * 8192),
    (torch.bfloat16, 500, 1024, 151936, 4096, 4096),         # a caller's smaller chunk is kept
    (torch.bfloat16, 500, 1024, 151936, 10000, 80128),       # 8 chunks, rounded up to tiles
    (torch.bfloat16, 16384, 2560, 151936, 8192, 8192),
])
def test_rows_staged_together(dtype, N, K, V, chunk, C):
    t = _lib.bwd_tiling(dtype, N, K, V, 64, chunk)
    assert t["C"] == C and t["n_chunks"] == -(-V // C), t
