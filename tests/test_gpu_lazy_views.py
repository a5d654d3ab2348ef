"""Tensors whose values the dispatcher still has to resolve (a sign to flip, zeros without memory) in
the calls that hand pointers to the library: the same results as from their plain copies.  One-element
tensors are the case, since ``.to`` and ``.contiguous()`` return them as they are."""
import pytest
import torch

import swvr_amd as swvr
from swvr_amd import _ops, fp8, vocab_shard
from tests.gpu_util import make


def negated(x):
    """``x``'s values as a lazily negated view (strided, as ``z.conj().imag`` is)."""
    out = torch.complex(torch.zeros_like(x), -x.detach().float()).conj().imag
    assert out.is_neg()
    return out


@pytest.mark.parametrize("zeros", [False, True])
def test_operands_are_resolved_before_their_pointers_are_taken(zeros):
    def lazy(*shape):
        return torch._efficientzerotensor(*shape) if zeros else negated(torch.ones(*shape))
    for n in (1, 9):
        for x in (_ops._f32(lazy(n)), _ops._f64(lazy(n, 1)), _ops._matrix(lazy(n, 8), torch.float32, 8),
                  _ops._operand(lazy(n, 8), torch.bfloat16, 8)[0], _ops._embed(lazy(n, 1), torch.float32)):
            assert not x.is_neg() and not x._is_zerotensor() and x.data_ptr() and (x == float(not zeros)).all()


def same(got, want):
    got, want = ([x for x in xs if x is not None] for xs in (got, want))
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float64])
def test_cotangents_of_one_token(dtype):
    xs = make(1, 40, 300, 1, dtype)
    gO, glse = torch.full((1, 1), 0.7, device="cuda"), torch.full((1,), 1.3, device="cuda")
    O, lse = swvr.softmax_readout(*xs)
    gO, glse = gO.to(O.dtype), glse.to(O.dtype)

    def lazy(x):
        return torch._neg_view(-x)
    grads = lambda a, b: torch.autograd.grad((O, lse), xs, (a, b), retain_graph=True)
    same(grads(lazy(gO), lazy(glse)), grads(gO, glse))
    z = torch._efficientzerotensor(1, dtype=O.dtype, device="cuda")
    same(grads(gO, z), grads(gO, torch.zeros_like(glse)))
    if dtype != torch.float64:
        a = (*[x.detach() for x in xs], O.detach(), lse.detach())
        same(vocab_shard.shard_backward(lazy(gO), lazy(glse), *a), vocab_shard.shard_backward(gO, glse, *a))


@pytest.mark.gpu
def test_the_loss_and_its_inputs():
    h, W, E, b = make(1, 40, 1, 1, torch.float32)
    target, weight, one = (torch.full(s, v, device="cuda") for s, v in (((1, 1), 2.5), ((1,), 0.5), ((1,), 0.3)))

    def call(target, weight, bias, E=E):
        xs = [h, W, E.detach().requires_grad_(True)]
        loss = swvr.softmax_readout_mse(*xs, target, bias, weight=weight, z_loss_weight=0.1, reduction="sum")
        return (loss, *torch.autograd.grad(loss, xs))
    same(call(negated(target), negated(weight), negated(one), negated(E)), call(target, weight, one))
    # the incoming gradient of a loss used as an imaginary part
    loss = lambda: swvr.softmax_readout_mse(h, W, E, target, b, weight=weight, reduction="none")
    got = torch.autograd.grad(loss(), (h, E), negated(one))
    same(got, torch.autograd.grad(loss(), (h, E), one))


@pytest.mark.gpu
def test_e4m3_cotangents_and_shard_partials():
    h, W, E, b = make(1, 64, 300, 1, torch.bfloat16)
    gO, glse = torch.full((1, 1), 0.7, device="cuda"), torch.full((1,), 1.3, device="cuda")
    O, lse = fp8.softmax_readout_fp8(h, W, E, b)
    grads = lambda a, c: torch.autograd.grad((O, lse), (h, W, E, b), (a, c), retain_graph=True)
    same(grads(negated(gO), negated(glse)), grads(gO, glse))
    m, l, acc = (torch.full(s, v, device="cuda") for s, v in (((1, 1), 1.5), ((1, 1), 2.0), ((1, 1, 1), 3.0)))
    same(vocab_shard.combine_partials(negated(m), negated(l), negated(acc)), vocab_shard.combine_partials(m, l, acc))
