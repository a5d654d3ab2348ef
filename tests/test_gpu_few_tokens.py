"""Calls with few tokens, whose kernels split their work differently from the large ones: every
output and gradient against the fp64 oracle.  Bars: the package's own, bf16 / fp16 1e-2 (O, lse) and
2e-2 (gradients), fp32 1e-5 (a fixed-order fp32 sum over at most 10^4 terms of either sign grows its
rounding error like sqrt(10^4) 2^-24 = 6e-6 at most)."""
import pytest
import torch

import swvr_amd as swvr
from tests.gpu_util import make, oracle_run, rel_err, run

pytestmark = pytest.mark.gpu


def check(inputs, fn, lead, D, bar_out, bar_grad):
    g = torch.Generator(device="cuda").manual_seed(7)
    gO = torch.randn(*lead, D, generator=g, device="cuda")
    glse = torch.randn(*lead, generator=g, device="cuda")
    out, ref = run(fn, inputs, gO, glse), oracle_run(inputs, gO, glse)
    errs = [rel_err(a, r) for a, r in zip(out, ref)]
    assert max(errs[:2]) <= bar_out and max(errs[2:]) <= bar_grad, errs


# dh tiles split over runs of a chunk's vocabulary rows: whole and ragged runs, a last chunk shorter
# than the runs (some of them empty), one chunk, a chunk of few slices (no split), a single token
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K,V,D,chunk,wrt_h", [
    (70, 264, 8232, 24, 8192, False),
    (300, 512, 6001, 64, 2048, False),
    (257, 256, 4096, 100, 4096, True),
    (1, 64, 3000, 16, 1024, False),
    (33, 300, 517, 40, 8192, True),
])
def test_dh_split_over_vocabulary_runs(dtype, N, K, V, D, chunk, wrt_h):
    h, W, E, b = make(N, K, V, D, dtype)
    if wrt_h:
        W, E, b = (x.detach() for x in (W, E, b))
    bars = (1e-2, 2e-2) if dtype == torch.bfloat16 else (1e-5, 1e-5)
    check((h, W, E, b), lambda *a: swvr.softmax_readout(*a, chunk_size=chunk), (N,), D, *bars)
