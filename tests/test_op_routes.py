"""The route of the differentiable ops: ordinary eager GPU calls run their kernels directly, everything
that observes or transforms an op (fake and meta tensors, tracing, tensor subclasses, function and dispatch
modes, functorch, forward mode) still gets the registered op; and the route of the one-process exchange."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from parallel_amd import ExpertPartition, TokenDispatcher, _lib, ops

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


class _Traced(torch.Tensor):
    """A tensor subclass that sees the functions called on it."""

    seen = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen.append(str(func))
        return super().__torch_function__(func, types, args, kwargs or {})


def _outcome(fn):
    """What a call does: its results, or the type of the exception that refuses it."""
    try:
        out = fn()
    except Exception as e:  # noqa: BLE001
        return type(e)
    return [o.detach() for o in (out if isinstance(out, tuple) else (out,))]


def _same(a, b):
    return a == b if isinstance(a, type) or isinstance(b, type) else (
        len(a) == len(b) and all(torch.equal(x, y) for x, y in zip(a, b)))


@pytest.mark.gpu
def test_the_direct_route_is_for_plain_eager_calls():
    """What decides, inside each of the situations that must not take it (private torch calls tell)."""
    x = torch.randn(4, 8, device="cuda")
    plain = ops._plain_eager
    assert plain((x, 2, True, None, 1.0)) and plain((torch.nn.Parameter(x),))
    assert not plain((x.as_subclass(_Traced),)) and not plain((x.cpu(),)) and not plain((x, "text"))
    seen = []

    def ask(t):
        seen.append(plain((x,)))
        return t.sum()

    torch.func.vmap(ask)(x)
    torch.func.grad(ask)(x)
    torch.func.jvp(ask, (x,), (x,))
    torch.func.functionalize(ask)(x)
    with torch.autograd.forward_ad.dual_level():
        ask(x)
    with _Seen():
        ask(x)
    with FakeTensorMode(allow_non_fake_inputs=True):
        seen.append(plain((x,)))
    torch.jit.trace(ask, (x,), check_trace=False)
    torch.fx.experimental.proxy_tensor.make_fx(ask)(x)
    with torch.overrides.BaseTorchFunctionMode():
        ask(x)
    assert len(seen) == 10 and not any(seen), seen
    assert plain((x,))  # and none of them leaves anything behind


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["subclass", "grad", "vjp", "vmap", "jvp", "forward_ad"])
def test_transformed_calls_do_what_the_registered_op_does(how):
    """The route under tensor subclasses, functorch transforms and forward mode: the registered op's
    results, or its refusal."""
    (x, rw, _, _), (k, norm) = _block_args(device="cuda")
    t = torch.ones_like(x)

    def call(op):
        f = lambda v: op(v, rw, k, norm)[1].float().square().sum()  # noqa: E731
        if how == "subclass":
            return op(x.as_subclass(_Traced), rw, k, norm)
        if how == "grad":
            return torch.func.grad(f)(x)
        if how == "vjp":
            out, back = torch.func.vjp(f, x)
            return out, *back(torch.ones_like(out))
        if how == "vmap":
            return torch.func.vmap(lambda v: op(v, rw, k, norm)[0])(x.unsqueeze(0))
        if how == "jvp":
            return torch.func.jvp(f, (x,), (t,))
        with torch.autograd.forward_ad.dual_level():
            return op(torch.autograd.forward_ad.make_dual(x, t), rw, k, norm)[0]

    _Traced.seen.clear()
    route = _outcome(lambda: call(ops.run_router_fwd))
    assert how != "subclass" or any("parallel_amd.router_fwd" in n for n in _Traced.seen)
    assert _same(route, _outcome(lambda: call(ops.router_fwd))), route


class _Recorded(TokenDispatcher):
    """A subclass with an exchange of its own."""

    def __init__(self, partition, group, extra=0):
        super().__init__(partition, group)
        self.modes, self.extra = [], extra

    def _exchange(self, value, send_splits, receive_splits, mode):
        self.modes.append(mode)
        return super()._exchange(value, send_splits, receive_splits, mode)

    def _exchange_splits(self, send_counts):
        send, receive = super()._exchange_splits(send_counts)
        return send, tuple(r + (self.extra if i == self.rank else 0) for i, r in enumerate(receive))


class _Splits(TokenDispatcher):
    def _exchange_splits(self, send_counts):
        send, receive = super()._exchange_splits(send_counts)
        return send, tuple(r + 1 for r in receive)


def test_own_block_route_is_for_the_dispatchers_own_exchange(monkeypatch):
    part = ExpertPartition(8, 2, 1)
    plain, patched = TokenDispatcher(part, None), TokenDispatcher(part, None)
    assert plain._exchanges_own_block() and not _Recorded(part, None)._exchanges_own_block()
    assert not TokenDispatcher(ExpertPartition(8, 1, 0), None)._exchanges_own_block()
    patched._exchange = lambda value, send, receive, mode: value
    assert not patched._exchanges_own_block()
    assert plain._is_own_block((3, 5), (0, 5), 8)
    for send, receive, rows in (((3, 5), (0, 5), 9), ((3, 5), (0, 4), 8), ((3, 5), (1, 5), 8), ((3, 5), (5,), 8)):
        assert not plain._is_own_block(send, receive, rows)
    monkeypatch.setattr("parallel_amd.groups.group_size", lambda group: 2)  # a group that grew after construction
    with pytest.raises(NotImplementedError):
        plain._exchanges_own_block()


@pytest.mark.gpu
def test_a_subclass_exchange_is_used():
    ids = torch.tensor([[0, 5], [6, 1], [7, 4]], device="cuda")
    hidden, scores = torch.randn(3, 64, device="cuda").to(BF), torch.rand(3, 2, device="cuda")
    part = ExpertPartition(8, 2, 1)
    recorded, plain = _Recorded(part, None), TokenDispatcher(part, None)
    got = recorded.dispatch(hidden, ids, scores)
    want = plain.dispatch(hidden, ids, scores)
    assert all(torch.equal(a, b) for a, b in zip(got[:3], want[:3]))
    assert torch.equal(recorded.combine(got[0], got[3]), plain.combine(want[0], want[3]))
    assert recorded.modes == ["dispatch_hidden", "dispatch_experts", "dispatch_scores", "combine_hidden"]
    for dispatcher in (_Recorded(part, None, extra=1), _Splits(part, None)):  # receive splits that don't match
        with pytest.raises(ValueError, match="expects"):
            dispatcher.dispatch(hidden, ids, scores)


def _dispatch_pass(T, E, k, H, ep, rank, layout):
    """Dispatch, an elementwise stand-in for the experts and combine, forward and backward."""
    g = torch.Generator().manual_seed(T + k)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).cuda()
    if layout == "none":  # no route of this rank
        ids = (ids % (E // ep) + ((rank + 1) % ep) * (E // ep))
    scores = torch.rand(T, k, generator=g).cuda().requires_grad_()
    hidden = torch.randn(T, H, generator=g).to(BF).cuda().requires_grad_()
    d_out = torch.randn(T, H, generator=g).to(BF).cuda()
    dispatcher = TokenDispatcher(ExpertPartition(E, ep, rank), None)
    received, experts, rscores, state = dispatcher.dispatch(hidden, ids, scores)
    rows = received * 1.5
    if layout == "strided":
        rows = torch.cat([rows, rows], dim=1)[:, :H]
    elif layout == "misaligned":
        rows = torch.cat([rows.new_zeros(3), rows.reshape(-1)])[3:].view(-1, H)
    out = dispatcher.combine(rows, state)
    grads = torch.autograd.grad([out, rscores], [hidden, scores], [d_out, torch.ones_like(rscores)])
    return [received.detach(), experts, rscores.detach(), state.source_tokens, state.pos_of_slot, out.detach(), *grads], (
        state.send_splits, state.receive_splits)


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,k,H,ep,rank,layout", [
    (1, 8, 1, 8, 2, 0, "plain"),          # one row of one 16-byte chunk
    (1, 8, 2, 2048, 4, 3, "plain"),
    (37, 16, 3, 264, 4, 1, "strided"),    # slot count at run time, a partial pass of the lanes
    (64, 128, 8, 2056, 2, 1, "plain"),    # 512 slots, the last size of the one-launch sort; one chunk past 2048
    (65, 128, 8, 512, 2, 0, "misaligned"),
    (300, 64, 6, 1536, 2, 1, "plain"),
    (33, 16, 16, 64, 4, 2, "plain"),
    (50, 16, 2, 128, 4, 2, "none"),
])
def test_own_block_exchange_gives_the_full_exchanges_bits(T, E, k, H, ep, rank, layout):
    got, splits = _dispatch_pass(T, E, k, H, ep, rank, layout)
    with _Seen() as seen:
        want, want_splits = _dispatch_pass(T, E, k, H, ep, rank, layout)
    assert any("combine_rows_fwd" in n for n in seen.names)
    assert splits == want_splits
    for i, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), f"result {i}"


@pytest.mark.gpu
def test_own_block_exchange_differentiates_twice():
    """Dispatch and combine are linear: the gradient as a function of d_out has the forward as its gradient."""
    ids = torch.tensor([[0, 5], [6, 1], [7, 4]], device="cuda")
    hidden = torch.randn(3, 64, device="cuda").to(BF).requires_grad_()
    d_out = torch.randn(3, 64, device="cuda").to(BF).requires_grad_()
    dispatcher = TokenDispatcher(ExpertPartition(8, 2, 1), None)
    received, _, _, state = dispatcher.dispatch(hidden, ids, torch.rand(3, 2, device="cuda"))
    (dh,) = torch.autograd.grad(dispatcher.combine(received, state), hidden, d_out, create_graph=True)
    (dd,) = torch.autograd.grad(dh, d_out, torch.ones_like(dh))
    count = torch.tensor([1, 1, 2], device="cuda").unsqueeze(1)
    assert torch.equal(dh, count * d_out) and torch.equal(dd, count.to(BF).expand(3, 64))


def test_block_entry_points_check_their_arguments():
    lib, buf = _lib.load(), torch.zeros(64, dtype=torch.int64)
    b = (buf.data_ptr() + 15) // 16 * 16
    for entry in (lib.moe_scatter_block, lib.moe_gather_block):
        assert entry(None, None, 0, 64, 2, 0, 0, None, None) == _lib.MOE_OK
        for T, H, k, lo, rows in ((2, 64, 2, 3, 2), (2, 64, 2, -1, 1), (2, 60, 2, 0, 1), (2, 64, 17, 0, 1)):
            assert entry(b, b, T, H, k, lo, rows, b, None) == _lib.MOE_ERR_INVALID
        assert entry(b, None, 2, 64, 2, 0, 1, b, None) == _lib.MOE_ERR_INVALID
        assert entry(b + 4, b, 2, 64, 2, 0, 1, b + 4, None) == _lib.MOE_ERR_INVALID
