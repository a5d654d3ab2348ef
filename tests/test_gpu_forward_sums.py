"""Sums of the forwards over long vocabularies, against 64 bits.  h and W are small multiples of powers of
two, so every score is exact in fp32 and what is measured is the softmax's own arithmetic."""
import pytest
import torch

import swvr_amd as swvr
from swvr_amd import vocab_shard as vs
from tests.gpu_util import rel_err

pytestmark = pytest.mark.gpu


def exact_scores(N, K, V, D, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    i = lambda lo, hi, *s: torch.randint(lo, hi + 1, s, generator=g, device="cuda").float()
    h, W, b = i(-4, 4, N, K) / 4, i(-8, 8, V, K) / 16, i(-64, 64, V) / 64
    return h.to(dtype), W.to(dtype), torch.randn(V, D, generator=g, device="cuda").to(dtype), b


def readout64(h, W, E, b):
    O, lse = [], []
    for x in h.split(512):
        S = x.double() @ W.double().T + b.double()
        lse.append(torch.logsumexp(S, -1))
        O.append(torch.exp(S.sub_(lse[-1][:, None])) @ E.double())
    return torch.cat(O), torch.cat(lse)


# The denominator l = sum e^(s - max) of a vocabulary shard: a run of it is summed in up to 300 steps, whose
# roundings (2.4e-8 rms each) add up to 2.4e-8 sqrt(300 / 3) = 2.4e-7 in one run and to an eighth of that or
# less over the 64 runs and more that are merged; e^x's own errors, up to 2^-21 each at the scores' spread,
# average out over the rows: 9e-8 measured, under 2^-23.  Scaled to another shift at every tile, by a factor
# that is itself rounded twice, l was 3.4e-7 (fp32, 8192 tokens) and 1.9e-7 (bf16, D = 128) off.
@pytest.mark.parametrize("dtype,N,D", [(torch.float32, 8192, 16), (torch.float32, 2000, 100), (torch.bfloat16, 8192, 64),
                                       (torch.bfloat16, 8192, 128), (torch.bfloat16, 768, 64), (torch.float16, 8192, 16)])
def test_sums_over_a_long_vocabulary(dtype, N, D):
    h, W, E, b = exact_scores(N, 64, 151936, D, dtype)
    m, l, _ = vs.softmax_readout_partial(h, W, E, b)
    O, lse = swvr.softmax_readout(h, W, E, b)
    rows = slice(0, N, 16)
    want_O, want_lse = readout64(h[rows], W, E, b)
    e_l = rel_err(l[rows].double() * torch.exp(m[rows].double() - want_lse), torch.ones_like(want_lse))
    e_lse, e_O = rel_err(lse[rows], want_lse), rel_err(O[rows], want_O)
    print(f"\n{dtype} {N}: l {e_l:.2e} lse {e_lse:.2e} O {e_O:.2e}")
    assert e_l <= 2 ** -23 and e_lse <= 2 ** -23 and e_O <= {torch.float32: 4e-6, torch.bfloat16: 1e-3,
                                                         torch.float16: 1.2e-4}[dtype]


# E near the largest finite values under scores that fall by 20 after the first row and, in the middle, rise
# again: no accumulator may pass what P <= 1 makes of them.  Vocabularies of several tiles per workgroup.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,V,D", [(40, 140001, 64), (700, 70001, 100), (1000, 20000, 64), (1000, 20000, 128),
                                   (1000, 20000, 256), (1000, 20000, 300)])
def test_embeddings_near_the_largest_finite_values(dtype, N, V, D):
    h, W = torch.zeros(N, 16, device="cuda", dtype=dtype), torch.zeros(V, 16, device="cuda", dtype=dtype)
    b = torch.zeros(V, device="cuda")
    b[0], b[V // 2], b[V // 2 + 1:V // 2 + 300] = 20, 15, -9
    E = torch.full((V, D), 2.0 ** 125, device="cuda", dtype=dtype)
    E[1::2] *= -1
    O, lse = swvr.softmax_readout(h, W, E, b)
    want_O, want_lse = readout64(h, W, E, b)
    assert rel_err(O, want_O) <= 1e-3 and rel_err(lse, want_lse) <= 1e-6


# scores that rise and fall by 40 over the vocabulary: shifts above, below and far below the running maximum
@pytest.mark.parametrize("dtype,bar", [(torch.bfloat16, 1e-3), (torch.float16, 2e-4), (torch.float32, 3e-6)])
@pytest.mark.parametrize("N,V,D,waves", [(3, 9001, 64, 3), (300, 40001, 33, 50), (700, 9001, 200, 7), (1500, 40001, 64, 40),
                                         (1500, 40001, 128, 40), (1500, 40001, 300, 9)])
def test_scores_that_rise_and_fall(dtype, bar, N, V, D, waves):
    h, W, E, _ = exact_scores(N, 64, V, D, dtype)
    b = 20 * torch.sin(torch.arange(V, device="cuda") * (2 * torch.pi * waves / V))
    O, lse = swvr.softmax_readout(h, W, E, b)
    want_O, want_lse = readout64(h, W, E, b)
    e_O, e_lse = rel_err(O, want_O), rel_err(lse, want_lse)
    print(f"\n{dtype} {N} {V} {D}: O {e_O:.2e} lse {e_lse:.2e}")
    assert e_O <= bar and e_lse <= 2 ** -23
