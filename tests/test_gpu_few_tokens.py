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


# the same merge where its 32 runs hold no, one or two partials each: a workgroup per 32 vocabulary rows,
# so V / 32 partials, and a merge of that many shards
@pytest.mark.parametrize("parts", [15, 16, 17, 31, 32, 33, 63, 64, 65])
def test_merge_of_few_partials(parts):
    from swvr_amd import vocab_shard as vs
    N, K, V, D = 7, 64, 32 * parts - 5, 40
    h, W, E, b = (x.detach() for x in make(N, K, V, D, torch.float32))
    b[32 * (parts - 2):] = float("-inf")   # the last two partials hold no score
    S = h.double() @ W.double().T + b.double()
    want_O, want_lse = torch.softmax(S, -1) @ E.double(), torch.logsumexp(S, -1)
    shards = [vs.softmax_readout_partial(h, W[v:v + 32], E[v:v + 32], b[v:v + 32]) for v in range(0, V, 32)]
    for O, lse in (swvr.softmax_readout(h, W, E, b), vs.combine_partials(*(torch.stack(x) for x in zip(*shards)))):
        assert rel_err(O, want_O) <= 1e-5 and rel_err(lse, want_lse) <= 1e-5


# the merge in 4 runs of 16 to 63 partials, up to 2^18 values (the third and fourth: both sides of that)
@pytest.mark.parametrize("N,V,D", [(1100, 12001, 100), (769, 6000, 97), (2048, 8001, 128), (2049, 8001, 128)])
def test_merge_of_some_partials(N, V, D):
    h, W, E, b = (x.detach() for x in make(N, 64, V, D, torch.float16))
    b[V // 3:2 * V // 3] = float("-inf")
    O, lse = swvr.softmax_readout(h, W, E, b)
    S = h.double() @ W.double().T + b.double()
    assert rel_err(O, torch.softmax(S, -1) @ E.double()) <= 1e-2 and rel_err(lse, torch.logsumexp(S, -1)) <= 1e-5


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


# the few-token forward: every token-block width, embedding width and storage type of it, sizes at the
# edges of its 32-token blocks, 128-row tiles, 128-byte slices and ring (short reductions), vocabularies
# of less than a group and of ragged runs, embeddings that need an aligned copy, several passes of columns
@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32", "autocast"])
@pytest.mark.parametrize("N,K,V,D", [
    (1, 72, 20011, 64), (31, 8, 97, 8), (32, 512, 9001, 200), (33, 40, 31, 128), (64, 1032, 5000, 33),
    (65, 264, 16385, 64), (128, 100, 4097, 72), (129, 96, 8193, 256), (255, 2048, 600, 300), (256, 64, 1, 16),
    (768, 64, 900, 64), (769, 136, 2000, 130),
])
def test_few_token_forward(dtype, N, K, V, D):
    amp = dtype == "autocast"
    dt = {"bf16": torch.bfloat16, "fp16": torch.float16}.get(dtype, torch.float32)
    h, W, E, b = make(N, K, V, D, dt, requires_grad=False)
    b[1:V // 3] = float("-inf")
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
        O, lse = swvr.softmax_readout(h, W, E, b, logit_scale=0.7)
    cd = torch.bfloat16 if amp else dt
    hd, Wd, Ed = (x.to(cd).double() for x in (h, W, E))
    S = 0.7 * (hd @ Wd.T) + b.double()
    want_O, want_lse = torch.softmax(S, -1) @ Ed, torch.logsumexp(S, -1)
    # P alone is rounded beside the operands: the rms of a rounding to 8 or 11 bits is 1.6e-3 or 2e-4, which
    # averages out over the rows but for the few that dominate; lse is a 32-bit sum
    bar = {torch.float32: 1e-5, torch.bfloat16: 2e-3, torch.float16: 2.5e-4}[cd]
    assert rel_err(O, want_O) <= bar and rel_err(lse, want_lse) <= 1e-5, (rel_err(O, want_O), rel_err(lse, want_lse))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_few_token_forward_equals_the_general_one_over_strides(dtype):
    """Strided h, W and E (row strides beyond their width, columns starting off 16 bytes) and a shard's
    partials: the same readout as from dense operands, and as rows of a call of many tokens."""
    from swvr_amd import vocab_shard as vs
    N, K, V, D = 40, 96, 3001, 48
    g = torch.Generator(device="cuda").manual_seed(5)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    h, W, E, b = r(300, K + 24)[:, 8:8 + K], r(V, K + 40)[:, 16:16 + K] / 8, r(V, D + 3)[:, 1:1 + D], r(V).float()
    O, lse = swvr.softmax_readout(h[:N], W, E, b)
    O_all, lse_all = swvr.softmax_readout(h, W, E, b)
    O_dense, lse_dense = swvr.softmax_readout(h[:N].contiguous(), W.contiguous(), E.contiguous(), b)
    assert torch.equal(O, O_dense) and torch.equal(lse, lse_dense)
    bar = 1e-5 if dtype == torch.float32 else 2e-3
    assert rel_err(O, O_all[:N]) <= bar and rel_err(lse, lse_all[:N]) <= 1e-5
    parts = [vs.softmax_readout_partial(h[:N], W[s], E[s], b[s]) for s in (slice(0, 1000), slice(1000, V))]
    O_s, lse_s = vs.combine_partials(*(torch.stack(x) for x in zip(*parts)))
    assert rel_err(O_s, O) <= bar and rel_err(lse_s, lse) <= 1e-5


def test_few_token_forward_keeps_non_finite_rows_apart():
    """An infinity or NaN in one token's h reaches that token alone, also where K ends inside a slice
    (the padding of h and W multiply to zero) and where the block holds other tokens."""
    N, K, V, D = 20, 40, 500, 16
    h, W, E, b = make(N, K, V, D, torch.bfloat16, requires_grad=False)
    h[3, 7], h[11, 39] = float("inf"), float("nan")
    O, lse = swvr.softmax_readout(h, W, E, b)
    bad = torch.zeros(N, dtype=torch.bool, device="cuda")
    bad[[3, 11]] = True
    assert O[bad].isnan().all() and O[~bad].isfinite().all() and lse[~bad].isfinite().all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N", [1, 128, 129, 512, 513])
def test_weighted_few_token_forward_zeroes_the_rows_of_zero_weight(dtype, N):
    """Both sides of the lines to the general active-token forward (128 in fp32, 512 else): the rows of
    non-zero weight as the unweighted call has them, zero rows for the others, a NaN column of E kept."""
    from swvr_amd import _ops
    K, V, D = 64, 700, 24
    h, W, E, b = make(N, K, V, D, dtype)
    w = (torch.arange(N, device="cuda") % 3 != 1).float()
    with torch.no_grad():
        O, lse = _ops._forward_active(h, W, E, b, w, 1.0, 8192, dtype)
        full = swvr.softmax_readout(h, W, E, b)
    on, bar = w != 0, 1e-5 if dtype == torch.float32 else 2e-3
    assert (O[~on] == 0).all() and (lse[~on] == 0).all()
    assert rel_err(O[on], full[0][on]) <= bar and rel_err(lse[on], full[1][on]) <= 1e-5
    bad = E.detach().clone()
    bad[V // 2, 3] = float("nan")
    O, lse = _ops._forward_active(h.detach(), W.detach(), bad, b.detach(), w, 1.0, 8192, dtype)
    assert O[:, 3].isnan().all() and (lse[on] != 0).all()


# embeddings wider than one pass whose last pass runs on a narrower kernel (64, 128 columns, whole
# passes beside), with token counts whose vocabulary splits are balanced and ones where they are not; in
# fp32 the passes are the few-token kernel's (the general kernels': the test of far-apart rows below)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("N,K,V,D", [(2500, 64, 9000, 300), (1100, 96, 3000, 257), (3000, 40, 4097, 640),
                                     (1030, 64, 300, 384)])
def test_last_pass_of_wide_embeddings_on_a_narrower_kernel(dtype, N, K, V, D):
    h, W, E, b = make(N, K, V, D, dtype, requires_grad=False)
    O, lse = swvr.softmax_readout(h, W, E, b)
    S = h.double() @ W.double().T + b.double()
    bar = 1e-5 if dtype == torch.float32 else 1e-2
    for sl in (slice(0, D // 256 * 256), slice(D // 256 * 256, D)):
        assert sl.start == sl.stop or rel_err(O[:, sl], torch.softmax(S, -1) @ E.double()[:, sl]) <= bar
    assert rel_err(lse, torch.logsumexp(S, -1)) <= bar


# rows of W or E further apart than the few-token kernel's 32-bit offsets reach (16 MB and more): packed for
# the general kernels, which fp32 and few tokens take for nothing else
@pytest.mark.parametrize("dtype,amp,N,D,far", [
    (torch.bfloat16, False, 20, 24, "W"), (torch.bfloat16, False, 200, 64, "E"), (torch.float16, False, 40, 300, "W"),
    (torch.float32, True, 33, 64, "W"), (torch.float32, False, 20, 24, "W"), (torch.float32, False, 300, 140, "W"),
    (torch.float32, False, 130, 64, "E")])
def test_rows_far_apart_take_the_general_kernels(dtype, amp, N, D, far):
    from swvr_amd import _ops
    K, V = 72, 130
    h, W, E, b = make(N, K, V, D, dtype, requires_grad=False)
    step = 2**24 // W.element_size() + 8   # 128 such rows: 2^31 bytes, the line
    x = W if far == "W" else E
    x2 = torch.empty((V - 1) * step + x.shape[1], dtype=dtype, device="cuda").as_strided(x.shape, (step, 1)).copy_(x)
    Wf, Ef = (x2, E) if far == "W" else (W, x2)
    weight = (torch.arange(N, device="cuda") % 3 > 0).float()

    def call(W, E):
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            cdt = torch.bfloat16 if amp else dtype
            return (*swvr.softmax_readout(h, W, E, b), *_ops._forward_active(h, W, E, b, weight, 1.0, 8192, cdt))
    bar = 1e-5 if dtype == torch.float32 and not amp else 2e-3
    for a, r in zip(call(Wf, Ef), call(W, E)):
        assert rel_err(a, r) <= bar


# the few-token kernel over the active tokens' positions (fp32 at any size, 2-byte types between 512 and
# 768 tokens): the device picks blocks and runs for the count, from none to all, at the edges of a block
@pytest.mark.parametrize("dtype,N", [(torch.float32, 2500), (torch.float32, 129), (torch.bfloat16, 700)])
@pytest.mark.parametrize("count", [0, 1, 127, 129, 10**6])
@pytest.mark.parametrize("V,D", [(3001, 20), (31, 140)])
def test_active_positions_on_the_few_token_kernel(dtype, N, count, V, D):
    from swvr_amd import _ops
    h, W, E, b = make(N, 72, V, D, dtype, requires_grad=False)
    w = torch.zeros(N, device="cuda")
    w[torch.randperm(N, generator=torch.Generator().manual_seed(1))[:count].cuda()] = 0.5
    O, lse = _ops._forward_active(h, W, E, b, w, 1.0, 8192, dtype)
    on = w != 0
    assert (O[~on] == 0).all() and (lse[~on] == 0).all()
    if count:
        S = h[on].double() @ W.double().T + b.double()
        bar = 1e-5 if dtype == torch.float32 else 1e-2
        assert rel_err(O[on], torch.softmax(S, -1) @ E.double()) <= bar
        assert rel_err(lse[on], torch.logsumexp(S, -1)) <= bar
    W2 = W.clone()
    W2[V - 1, 71] = float("nan")   # a parameter's NaN keeps every token computed, as the reference's loss needs
    O, lse = _ops._forward_active(h, W2, E, b, w, 1.0, 8192, dtype)
    assert O.isnan().all() and lse.isnan().all()


# no chunk given: several times 8192 rows staged together, and a second such group that is not whole
@pytest.mark.parametrize("dtype,N,K,V,D", [(torch.bfloat16, 200, 64, 270001, 24),
                                           (torch.bfloat16, 1030, 72, 40000, 100), (torch.float32, 520, 64, 66000, 16)])
def test_chunks_staged_together(dtype, N, K, V, D):
    inputs = make(N, K, V, D, dtype, w_scale=1.0)
    bars = (1e-2, 2e-2) if dtype == torch.bfloat16 else (1e-5, 1e-5)
    from swvr_amd import _lib, _ops
    tag = _lib.DTYPE_TAG[dtype]
    rows = _ops._rows_staged(None, tag, tag, N, (K + 7) // 8 * 8, V, D, True)
    assert 8192 < rows < V
    check(inputs, swvr.softmax_readout, (N,), D, *bars)


@pytest.mark.parametrize("chunk", [8192, None])
def test_backward_memory_of_few_tokens(chunk):
    """Beyond the gradients: a given chunk's workspace (69 MiB here), or without one at most what 8192 tokens
    take at 8192 rows (294 MiB) and 64 MiB; 10 MiB for the rest of the call."""
    N, K, V, D = 500, 1024, 151936, 64
    xs = make(N, K, V, D, torch.bfloat16)
    loss = swvr.softmax_readout_mse(*xs[:3], torch.randn(N, D, device="cuda"), xs[3], chunk_size=chunk)
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    grads = torch.autograd.grad(loss, xs)
    torch.cuda.synchronize()
    extra = (torch.cuda.max_memory_allocated() - base - sum(g.numel() * g.element_size() for g in grads)) / 2**20
    print(f"{extra:.0f} MiB")
    assert extra <= (69 if chunk else 294 + 64) + 10
