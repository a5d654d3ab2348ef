"""How many vocabulary rows a backward stages at a time (no GPU needed): a chunk that is given is kept and
bounds the workspace; without one, up to 4096 tokens take a power of two of chunks of 8192 rows, within
the workspace that 8192 tokens take at one."""
import pytest
import torch

import swvr_amd
from swvr_amd import _lib, _ops, api

BF, F32 = torch.bfloat16, torch.float32


def workspace(dtype, w_dtype, N, K, V, D, chunk, need_gh=1):
    tag = _lib.DTYPE_TAG
    return _lib.load().swvr_bwd_workspace_size_mixed(tag[dtype], tag[w_dtype], N, K, V, D, chunk, need_gh)


def default_rows(dtype, w_dtype, N, K, V, D, need_gh=1):
    return _ops._rows_staged(None, _lib.DTYPE_TAG[dtype], _lib.DTYPE_TAG[w_dtype], N, K, V, D, need_gh)


@pytest.mark.parametrize("N,K,V,chunk,C", [
    (500, 1024, 151936, 8192, 8192), (500, 1024, 151936, 16384, 16384), (500, 1024, 151936, 4096, 4096),
    (500, 1024, 151936, 10000, 10240), (1, 256, 10**6, 8192, 8192), (500, 1024, 6000, 8192, 6144),
    (16384, 2560, 151936, 8192, 8192),
])
def test_a_given_chunk_is_kept(N, K, V, chunk, C):
    t = _lib.bwd_tiling(BF, N, K, V, 64, chunk)
    assert t["C"] == C and t["n_chunks"] == -(-V // C), t


SIZES = [(1024, 151936, 64), (256, 256000, 300), (2048, 65536, 128), (768, 30001, 100), (4096, 256000, 256),
         (1024, 32000, 16)]


@pytest.mark.parametrize("dtype,w_dtype", [(BF, BF), (BF, F32), (F32, F32)])
@pytest.mark.parametrize("K,V,D", SIZES)
def test_a_given_chunk_bounds_the_workspace(dtype, w_dtype, K, V, D):
    """What is held per row of a chunk: dS and, for wide embeddings, P over the padded tokens, twice that at
    most for partial sums of gh, packed W (and the rounded rows of an fp32 W for two chunks), dE and db
    partials of at most 32 (256 / 8) groups; beside it the packed E and what is held per token."""
    b = 2 if dtype == BF else 4
    for N in (1, 256, 500, 1024, 4096):
        pad, DP = -(-N // 256) * 256, -(-D // 32) * 32
        for chunk in (256, 1024, 8192, 16384):
            C = min(chunk, V) + 256
            parts = min(256, -(-256 * 256 // C), -(-N // 32))
            per_row = 4 * pad * b + (K + 64) * b * (3 if dtype != w_dtype else 1) + 2 * parts * (DP + 1) * 4
            per_token = 3 * K * b + K * 4 + 2 * DP * b + 64
            bound = C * per_row + (V + 256) * (DP * b + 4) + pad * per_token + 2**16
            assert workspace(dtype, w_dtype, N, K, V, D, chunk) <= bound, (N, chunk)


@pytest.mark.parametrize("need_gh", [0, 1])
@pytest.mark.parametrize("dtype,w_dtype", [(BF, BF), (BF, F32), (F32, F32)])
@pytest.mark.parametrize("K,V,D", SIZES)
def test_the_default_stays_within_the_workspace_of_8192_tokens(dtype, w_dtype, K, V, D, need_gh):
    most = workspace(dtype, w_dtype, 8192, K, V, D, 8192, need_gh) + need_gh * 2**26
    for N in (1, 255, 256, 257, 500, 1000, 1024, 1025, 2048, 2049, 4096):
        rows = default_rows(dtype, w_dtype, N, K, V, D, need_gh)
        n = rows // 8192
        assert rows == n * 8192 and n & (n - 1) == 0 and 1 <= n <= 32 and n * -(-N // 256) * 256 <= 8192
        assert n == 1 or (n // 2) * 8192 < V
        assert workspace(dtype, w_dtype, N, K, V, D, rows, need_gh) <= most, (N, rows)
    for N in (4097, 8192, 16384):
        assert default_rows(dtype, w_dtype, N, K, V, D, need_gh) == 8192


@pytest.mark.parametrize("dtype,w_dtype,N,K,V,D,n", [
    (BF, BF, 500, 1024, 32000, 64, 4), (BF, BF, 500, 1024, 151936, 64, 8), (BF, F32, 500, 1024, 151936, 64, 4),
    (BF, BF, 2048, 1024, 151936, 16, 4), (BF, BF, 4096, 1024, 128256, 64, 2), (F32, F32, 1332, 768, 30001, 100, 4),
    (BF, F32, 2048, 2048, 65536, 128, 2), (F32, F32, 512, 256, 4096, 16, 1),
])
def test_the_default_at_some_sizes(dtype, w_dtype, N, K, V, D, n):
    assert default_rows(dtype, w_dtype, N, K, V, D) == n * 8192


def test_where_the_chunk_comes_from(monkeypatch):
    monkeypatch.delenv("SWVR_CHUNK", raising=False)
    assert api._chunk(None) is None and api._chunk(0) is None and api._chunk(8192) == 8192
    monkeypatch.setenv("SWVR_CHUNK", "8192")
    assert api._chunk(None) == 8192 and api._chunk(512) == 512
    assert _ops._rows_staged(8192, 0, 0, 1, 64, 10**6, 16, True) == 8192
    monkeypatch.setenv("SWVR_CHUNK", "-4")
    x = torch.empty(2, 8, device="meta")
    for size in (None, -1):
        with pytest.raises(ValueError, match="chunk_size must be positive"):
            swvr_amd.softmax_readout(x, x, x, chunk_size=size)
    lib = _lib.load()
    assert lib.swvr_bwd_default_chunk(9, 9, 1, 8, 0, 8, 8, 1) == 0
    assert lib.swvr_bwd_default_chunk(0, 0, -1, 8, 0, 8, 8, 1) == 0
    assert lib.swvr_bwd_default_chunk(0, 0, 0, 8, 0, 10**6, 8, 1) == 8192
    assert lib.swvr_bwd_default_chunk(0, 0, 500, 1024, 1024, 151936, 64, 1) > 8192      # e4m3 scores
