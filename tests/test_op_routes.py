"""The route of the differentiable ops: ordinary eager GPU calls run their kernels directly, everything
that observes or transforms an op (fake and meta tensors, symbolic tracing, tensor subclasses, dispatch
modes, functorch) still gets the registered op."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from parallel_amd import ops

BF = torch.bfloat16


def _block_args(T=64, H=128, E=16, I=64, k=4, device="cpu", **kw):
    g = torch.Generator().manual_seed(3)

    def t(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(BF).to(device)

    return [t(T, H), t(E, H, std=0.1), t(E, 2 * I, H, std=0.05), t(E, H, I, std=0.05)], (k, True)


@pytest.mark.parametrize("grad", [False, True])
def test_fake_and_meta_tensors_get_the_registered_op(grad):
    with FakeTensorMode():
        (x, rw, gu, dn), rest = _block_args(device="cuda" if torch.cuda.is_available() else "cpu")
        leaves = [v.requires_grad_(grad) for v in (x, rw, gu, dn)]
        out, logits, scores, idx, aux = ops.moe_block(*leaves, *rest)
        assert out.shape == x.shape and logits.shape == (64, 16) and idx.dtype == torch.int64
        assert type(out).__name__ == "FakeTensor" and out.requires_grad == grad
    (x, rw, _, _), rest = _block_args()
    out = ops.run_router_fwd(x.to("meta"), rw.to("meta"), *rest)
    assert out[0].device.type == "meta" and out[0].shape == (64, 16)


def test_symbolic_tracing_records_the_op():
    traced = torch.fx.symbolic_trace(lambda x, w: ops.run_router_fwd(x, w, 4, True))
    assert any(n.target is torch.ops.parallel_amd.router_fwd.default for n in traced.graph.nodes)


def test_cpu_tensors_are_refused_as_before():
    (x, rw, gu, dn), rest = _block_args()
    with pytest.raises(ValueError, match="GPU only"):
        ops.moe_block(x, rw, gu, dn, *rest)


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("mode", ["no_grad", "inference", "grad"])
def test_direct_calls_give_the_ops_bits(mode, dtype):
    """moe_block, experts, the router, the norm and the aux loss: direct against the registered ops
    (which a dispatch mode around the call selects), values and gradients."""
    args, (k, norm) = _block_args(device="cuda")
    args = [a.to(dtype) for a in args]

    def results():
        x, rw, gu, dn = [a.clone().requires_grad_(mode == "grad") for a in args]
        out, logits, scores, idx, aux = ops.moe_block(x, rw, gu, dn, k, norm)
        got = [out, logits, scores, idx, aux]
        router = ops.run_router_aux_fwd(x, rw, k, norm, None, None)
        out2 = ops.experts(x, router[2], router[1], gu, dn)
        got += [*router, out2]
        loss = out.float().square().sum() + aux + out2.float().sum() + router[3]
        if dtype == BF:
            gamma = torch.ones(x.shape[1], dtype=BF, device="cuda", requires_grad=mode == "grad")
            h, rstd = ops.run_rmsnorm_fwd(x.view(4, 16, -1), gamma, 1e-6)
            sent = ops.run_dispatch_fwd(x, idx, router[1], 8, 2)
            back = ops.run_combine_rows_fwd(sent[0], sent[4], x.shape[0], k)
            got += [h, rstd, *sent, back]
            loss = loss + h.float().square().sum() + back.float().sum()
        if mode == "grad":
            loss.backward()
            got += [v.grad for v in (x, rw, gu, dn)] + ([gamma.grad] if dtype == BF else [])
        return [g.detach() for g in got]

    ctx = {"no_grad": torch.no_grad, "inference": torch.inference_mode, "grad": torch.enable_grad}[mode]
    with ctx():
        direct = results()
        with _Seen() as seen:
            through_ops = results()
    assert any("parallel_amd.moe_block_fwd" in n for n in seen.names)
    assert len(direct) == len(through_ops)
    for i, (a, b) in enumerate(zip(direct, through_ops)):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), f"result {i}"


@pytest.mark.gpu
def test_direct_calls_keep_hooks_and_in_place_outputs():
    args, (k, norm) = _block_args(device="cuda")
    x, rw, gu, dn = [a.requires_grad_() for a in args]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t)[1], lambda t: t):
        out = ops.moe_block(x, rw, gu, dn, k, norm)[0]
    assert torch.Size(gu.shape) in packed
    h, _ = ops.run_rmsnorm_fwd(x.view(4, 16, -1), torch.ones(x.shape[1], dtype=BF, device="cuda"), 1e-6)
    h += 1  # a fresh tensor, not a view: in-place use stays legal
    (out.float().sum() + h.float().sum()).backward()
    assert all(v.grad is not None for v in (x, rw, gu, dn))
