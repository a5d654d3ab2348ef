"""Plain eager calls, which go to the library as one autograd node, against the same calls through the
custom ops (which any active function mode selects): equal bits, and the ops seen by whatever looks at
them."""
import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

import swvr_amd as swvr
from swvr_amd import _ops
from tests.gpu_util import make

pytestmark = pytest.mark.gpu


class ThroughOps(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class SeenOps(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = set()

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.add(str(func))
        return func(*args, **(kwargs or {}))


def loss_and_grads(xs, target, weight, **kw):
    h, W, E, b = xs
    out = swvr.softmax_readout_mse(h, W, E, target, b, weight=weight, **kw)
    return (out, *torch.autograd.grad(out.sum(), [x for x in xs if x is not None and x.requires_grad]))


@pytest.mark.parametrize("reduction", ["none", "sum", "mean"])
@pytest.mark.parametrize("lead,weighted,bias,frozen", [((70,), True, True, ()), ((3, 40), True, False, (0,)),
                                                       ((2, 5, 7), False, True, (1, 2)), ((), False, True, ())])
def test_mse_node_equals_the_ops(reduction, lead, weighted, bias, frozen):
    K, V, D = 72, 901, 24
    xs = make(1, K, V, D, torch.bfloat16, bias=bias, lead=lead or (1,))
    if not lead:
        xs[0] = xs[0].detach()[0].requires_grad_(True)
    for i in frozen:
        xs[i] = xs[i].detach()
    target = torch.randn(*lead, D, device="cuda")
    weight = (torch.arange(target[..., 0].numel(), device="cuda") % 3 > 0).float().view(lead) if weighted else None
    kw = dict(reduction=reduction, z_loss_weight=1e-3, logit_scale=0.5, chunk_size=256)
    got = loss_and_grads(xs, target, weight, **kw)
    with ThroughOps():
        want = loss_and_grads(xs, target, weight, **kw)
    assert got[0].grad_fn.name().startswith(("_ReadoutMse", "View", "Alias")) and got[0].shape == want[0].shape
    for a, r in zip(got, want):
        assert a.dtype == r.dtype and torch.equal(a, r)
    with torch.no_grad():
        assert torch.equal(swvr.softmax_readout_mse(*xs[:3], target, xs[3], weight=weight, **kw), got[0])


@pytest.mark.parametrize("used", ["O", "lse", "both"])
def test_readout_node_equals_the_ops(used):
    xs = make(50, 72, 901, 24, torch.float32)

    def run():
        O, lse = swvr.softmax_readout(*xs, chunk_size=256)
        y = {"O": O.sin().sum(), "lse": lse.cos().sum(), "both": O.sin().sum() + lse.cos().sum()}[used]
        return (O, lse, *torch.autograd.grad(y, xs))
    got = run()
    with ThroughOps():
        want = run()
    for a, r in zip(got, want):
        assert torch.equal(a, r)


def test_whatever_looks_at_the_ops_sees_them():
    xs = make(20, 64, 300, 16, torch.float32)
    target, weight = torch.randn(20, 16, device="cuda"), torch.ones(20, device="cuda")
    with SeenOps() as seen:
        swvr.softmax_readout(*xs)
        swvr.softmax_readout_mse(*xs[:3], target, xs[3], weight=weight)
    assert {"swvr.chunked_fwd.default", "swvr.chunked_fwd_active.default", "swvr.mse_loss.default"} <= seen.names
    assert not _ops.eager(xs[0].cpu()) and _ops.eager(xs[0], None)

    def inside(x):
        assert not _ops.eager(x.detach())
        return x.sum()
    torch.func.grad(inside)(xs[0].detach())
    with torch.autograd.forward_ad.dual_level():
        assert not _ops.eager(xs[0])


@pytest.mark.parametrize("loss", ["readout", "mse", "weighted"])
def test_a_backward_run_under_a_mode_shows_its_op(loss):
    xs = make(20, 64, 300, 16, torch.float32)
    xs[1].requires_grad_(False)
    target, weight = torch.randn(20, 16, device="cuda"), (torch.arange(20, device="cuda") % 4 > 0).float()

    def run():
        if loss == "readout":
            O, lse = swvr.softmax_readout(*xs, chunk_size=256)
            return O.sin().sum() + lse.cos().sum()
        w = weight if loss == "weighted" else None
        return swvr.softmax_readout_mse(*xs[:3], target, xs[3], weight=w, chunk_size=256)
    wrt = [xs[0], xs[2], xs[3]]
    want, out = torch.autograd.grad(run(), wrt), run()
    with SeenOps() as seen:
        got = torch.autograd.grad(out, wrt)
    assert "swvr.chunked_bwd.default" in seen.names and "swvr.chunked_fwd.default" not in seen.names
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_calls_without_a_chunk_agree_compiled_and_eager():
    """Eager calls of few tokens stage more rows at a time than the ops' 8192, compiled ones those: the same
    gradients but for the order of gh's sums."""
    xs = make(40, 64, 20000, 16, torch.float32)
    target = torch.randn(40, 16, device="cuda")
    fn = lambda h: swvr.softmax_readout_mse(h, *xs[1:3], target, xs[3])
    torch._dynamo.reset()
    loss_c, loss_e = torch.compile(fn, fullgraph=True)(xs[0]), fn(xs[0])
    assert _ops._rows_staged(None, 2, 2, 40, 64, 20000, 16, True) > 8192
    assert torch.equal(loss_c, loss_e)
    for a, b in zip(torch.autograd.grad(loss_c, xs), torch.autograd.grad(loss_e, xs)):
        assert (a - b).norm() <= 1e-5 * b.norm()


def test_saved_tensor_hooks_and_a_second_derivative():
    xs = make(20, 64, 300, 16, torch.float32)
    target = torch.randn(20, 16, device="cuda")
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        loss = swvr.softmax_readout_mse(*xs[:3], target, xs[3])
    want = torch.autograd.grad(swvr.softmax_readout_mse(*xs[:3], target, xs[3]), xs)
    assert packed and all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(loss, xs), want))
    g, = torch.autograd.grad(swvr.softmax_readout_mse(*xs[:3], target, xs[3]), xs[:1], create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g.sum(), xs[:1])
    loss = swvr.softmax_readout_mse(*xs[:3], target, xs[3])
    with torch.no_grad():
        xs[1].add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(loss, xs[:1])
