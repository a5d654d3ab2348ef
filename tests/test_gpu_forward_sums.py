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
    assert e_l <= 2 ** -23 and e_lse <= 2 ** -23 and e_O <= {torch.float32: 4e-6, torch.bfloat16: 1.2e-3,
                                                         torch.float16: 1.5e-4}[dtype]
