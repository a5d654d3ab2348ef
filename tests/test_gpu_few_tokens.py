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


# the merge of many partial softmaxes in 32 runs (few tokens, a long vocabulary) and in 8 (few
# partials): rows with every score -inf, whole partials of -inf, and embedding widths off the tiles
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K,V,D", [(1, 40, 70001, 1), (31, 64, 70001, 40), (33, 64, 9000, 33), (700, 64, 2048, 129)])
def test_merge_of_partials(dtype, N, K, V, D):
    h, W, E, b = make(N, K, V, D, dtype)
    with torch.no_grad():
        b[V // 4:3 * V // 4] = float("-inf")
    bars = (1e-2, 2e-2) if dtype == torch.bfloat16 else (1e-5, 1e-5)
    check((h, W, E, b), swvr.softmax_readout, (N,), D, *bars)
    O, lse = swvr.softmax_readout(h.detach(), W.detach(), E.detach(), torch.full_like(b.detach(), float("-inf")))
    assert O.isnan().all() and (lse == float("-inf")).all()


@pytest.mark.parametrize("N", [1, 1023, 1024, 1025, 4097, 300001])
def test_compaction_of_active_tokens_over_workgroups(N):
    """Weights of 0 drop tokens; the others keep their own rows: sizes at the edges of a workgroup's
    1024 tokens and past 256 workgroups' worth, with a whole workgroup's tokens dropped."""
    K, V, D = 8, 40, 8
    h, W, E, b = make(N, K, V, D, torch.float32)
    g = torch.Generator(device="cuda").manual_seed(3)
    w = (torch.rand(N, generator=g, device="cuda") < 0.4).float()
    w[2048:3072] = 0
    t = torch.randn(N, D, generator=g, device="cuda")
    loss = swvr.softmax_readout_mse(h, W, E, t, b, weight=w, reduction="none")
    got = torch.autograd.grad(loss.sum(), (h, W))
    ref = [x.detach().double().requires_grad_(True) for x in (h, W)]
    O = torch.softmax(ref[0] @ ref[1].T + b.detach().double(), -1) @ E.detach().double()
    want_loss = (O - t.double()).pow(2).mean(-1) * w.double()
    want = torch.autograd.grad(want_loss.sum(), ref)
    if not w.any():
        assert (loss == 0).all() and all((x == 0).all() for x in got)
        return
    # gW sums n terms of either sign in fp32: its partial sums grow like sqrt(k), so the roundings
    # add up to about sqrt(sum k) 2^-24 against a sum of sqrt(n), sqrt(n / 2) 2^-24; twice that
    errs = [rel_err(a, r) for a, r in zip((loss, *got), (want_loss, *want))]
    assert max(errs[:2]) <= 1e-5 and errs[2] <= max(1e-5, w.sum().item() ** 0.5 * 2 ** -23.5), errs
    assert (got[0][w == 0] == 0).all()
