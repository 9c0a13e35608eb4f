"""What the operators owe autograd because their nodes are native: the things torch.autograd.Function does for an operator
written in Python.  On the CPU through the x86 build of the kernels, on the GPU through the library."""
import contextlib

import pytest
import torch
import torch.autograd.forward_ad as fwAD

import llsa_amd
from emu_util import emu_lib
from llsa_amd._lib import override_library_for_tests


@pytest.fixture(params=["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def dev(request):
    with contextlib.ExitStack() as stack:
        if request.param == "cpu":
            stack.enter_context(override_library_for_tests(emu_lib()))
        yield torch.device(request.param)


def _inputs(dev, n=3, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(1, 1, 1024, 64, generator=g).bfloat16().to(dev) for _ in range(n)]


def _permutation(dev, n=64):
    perm = torch.randperm(n, generator=torch.Generator().manual_seed(1))
    return perm.int().to(dev), torch.argsort(perm).int().to(dev)


@pytest.mark.parametrize("which", ["q", "k", "v", "rope", "gamma_q", "gamma_k", "tokens"])
def test_tangents_are_refused(dev, which):
    """An input that carries a tangent is an error: the kernels have no forward-mode rule."""
    q, k, v = _inputs(dev)
    rope, gq, gk = torch.zeros(1024, 64, device=dev).bfloat16(), torch.ones(64, device=dev), torch.ones(64, device=dev)
    x, (perm, inv) = torch.randn(1, 64, 8, device=dev), _permutation(dev)
    with fwAD.dual_level():
        dual = lambda name, t: fwAD.make_dual(t, torch.ones_like(t)) if name == which else t
        for mode in (contextlib.nullcontext(), torch.no_grad()):
            with mode, pytest.raises(NotImplementedError, match="jvp"):
                if which == "tokens":
                    llsa_amd.permute_tokens(dual("tokens", x), perm, inv)
                else:
                    llsa_amd.llsa_l1(dual("q", q), dual("k", k), dual("v", v), 8, 16, rope=dual("rope", rope),
                                     qk_norm=(dual("gamma_q", gq), dual("gamma_k", gk), 1e-5))


def test_function_transforms_are_refused(dev):
    q, k, v = _inputs(dev)
    x, (perm, inv) = torch.randn(1, 64, 8, device=dev), _permutation(dev)
    permute = lambda a: llsa_amd.permute_tokens(a, perm, inv)
    for call in (lambda: torch.func.vmap(permute)(x[None]), lambda: torch.func.grad(lambda a: permute(a).sum())(x),
                 lambda: torch.func.jvp(permute, (x,), (x,)), lambda: torch.func.grad(lambda s: (permute(x) * s).sum())(torch.ones((), device=dev)),
                 lambda: torch.func.vmap(lambda a: llsa_amd.llsa_l1(a, k, v, 8, 16))(q[None])):
        with pytest.raises(RuntimeError, match="functorch transforms"):
            call()


def _operator(norm, rope):
    def fn(q, k, v, gq, gk, freq):
        return llsa_amd.llsa_l1(q, k, v, 8, 16, rope=freq if rope else None, qk_norm=(gq, gk, 1e-5) if norm else None)
    return fn


def _leaves(dev):
    q, k, v = (t.requires_grad_() for t in _inputs(dev))
    gq, gk = (torch.linspace(0.5, 1.5, 64, device=dev).requires_grad_() for _ in range(2))
    freq = torch.randn(1024, 64, generator=torch.Generator().manual_seed(5)).bfloat16().to(dev)
    return [q, k, v, gq, gk], freq


def _same_gradients(run, reference, do):
    """run and reference: functions of nothing that return (output, leaves); gradients compared bit for bit."""
    grads = []
    for fn in (run, reference):
        o, leaves = fn()
        used = [t for t in leaves if t.grad_fn is None]
        grads.append((o.detach(), torch.autograd.grad(o, used, do, allow_unused=True)))
    assert torch.equal(grads[0][0], grads[1][0])
    for a, b in zip(grads[0][1], grads[1][1]):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


@pytest.mark.parametrize("norm,rope", [(False, False), (True, True)])
def test_saved_tensor_hooks_see_everything(dev, norm, rope):
    """All that the forward keeps passes through the hooks, packed into copies that are unaligned and elsewhere in memory."""
    fn, do = _operator(norm, rope), torch.randn(1, 1, 1024, 64, generator=torch.Generator().manual_seed(9)).bfloat16().to(dev)
    packed = []

    def pack(t):
        packed.append(t.numel() * t.element_size())
        room = torch.empty(t.numel() + 1, dtype=t.dtype, device="cpu")
        room[1:] = t.detach().reshape(-1).cpu()
        return room, t.shape

    def unpack(p):
        return p[0].to(dev)[1:].view(p[1])

    def hooked():
        leaves, freq = _leaves(dev)
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            return fn(*leaves, freq), leaves

    def plain():
        leaves, freq = _leaves(dev)
        return fn(*leaves, freq), leaves

    _same_gradients(hooked, plain, do)
    tiles = 3 * 1024 * 64 * 2                                 # the operand tiles of q, k, v alone; then o, lse, selection, lists
    assert sum(packed) >= tiles + 1024 * 64 * 2 + 4 * 1024 + 2 * 4 * 64 * 8


def test_saved_tensors_on_the_host(dev):
    do = torch.ones(1, 1, 1024, 64, device=dev).bfloat16()

    def run(ctx):
        def go():
            leaves, freq = _leaves(dev)
            with ctx():
                return _operator(False, True)(*leaves, freq), leaves
        return go
    _same_gradients(run(lambda: torch.autograd.graph.save_on_cpu()), run(contextlib.nullcontext), do)


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("reentrant", [False, True])
def test_checkpoint(dev, norm, reentrant):
    """A checkpointed block around the operator, whose recomputation runs inside the operator's own backward."""
    from torch.utils.checkpoint import checkpoint
    w = torch.randn(64, 64, generator=torch.Generator().manual_seed(3)).bfloat16().to(dev) / 8
    do = torch.randn(1, 1, 1024, 64, generator=torch.Generator().manual_seed(9)).bfloat16().to(dev)

    def run(use):
        def go():
            leaves, freq = _leaves(dev)
            wl = w.clone().requires_grad_()
            block = lambda q, k, v, gq, gk: _operator(norm, True)(q @ wl, k @ wl, v, gq, gk, freq) * 2
            return (checkpoint(block, *leaves, use_reentrant=reentrant) if use else block(*leaves)), leaves + ([wl] if not reentrant else [])
        return go
    if reentrant:                                             # (only .backward() works there)
        grads = []
        for use in (True, False):
            o, leaves = run(use)()
            o.backward(do)
            grads.append([t.grad for t in leaves])
        assert all((a is None) == (b is None) and (a is None or torch.equal(a, b)) for a, b in zip(*grads))
    else:
        _same_gradients(run(True), run(False), do)


def test_selection_through_hooks(dev):
    from llsa_amd.kernel.torch_op._fused import selection
    leaves, _ = _leaves(dev)
    plain = selection(llsa_amd.llsa_l1(*leaves[:3], 8, 16))[0]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(dev)):
        o = llsa_amd.llsa_l1(*leaves[:3], 8, 16)
    assert torch.equal(selection(o)[0], plain)


def test_a_hook_that_returns_another_tensor_is_an_error(dev):
    leaves, _ = _leaves(dev)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.reshape(-1)[:64] if t.dtype == torch.uint8 else t):
        o = llsa_amd.llsa_l1(*leaves[:3], 8, 16)
    with pytest.raises(RuntimeError, match="another tensor"):
        o.backward(torch.ones_like(o))


@pytest.mark.parametrize("grad", [False, True])
def test_trace(dev, grad):
    """A traced permutation computes, on other inputs too; the attention operators refuse to be traced."""
    x, y = (torch.randn(2, 64, 8, generator=torch.Generator().manual_seed(s)).to(dev).requires_grad_(grad) for s in (1, 2))
    perm, inv = _permutation(dev)
    traced = torch.jit.trace(lambda a: llsa_amd.permute_tokens(a * 2, perm, inv), (x,), check_trace=False)
    got, ref = traced(y), 2 * y.detach()[:, perm.long(), :]
    assert torch.equal(got, ref)
    if grad:
        got.backward(ref)
        assert torch.equal(y.grad, 4 * y.detach())
    q, k, v = _inputs(dev)
    with pytest.raises(RuntimeError, match="torch.jit.trace"):
        torch.jit.trace(lambda a: llsa_amd.llsa_l1(a, k, v, 8, 16), (q,), check_trace=False)


def test_arguments(dev):
    """Any block_size that equals 16 is one; errors name dtypes as torch does; a permutation that is never differentiated needs
    no inverse."""
    import numpy as np
    q, k, v = _inputs(dev)
    for size in (16.0, np.int64(16), torch.tensor(16)):
        assert llsa_amd.llsa_l1(q, k, v, 8, size).shape == q.shape
    for size in (8, None):
        with pytest.raises(NotImplementedError, match="block_size must be 16"):
            llsa_amd.llsa_l1(q, k, v, 8, size)
    for dtype in (torch.float64, torch.float32, torch.float16, torch.int64, torch.bool, torch.float8_e4m3fn):
        with pytest.raises(NotImplementedError, match=f"got {dtype}"):
            llsa_amd.llsa_l1(q.to(dtype), k, v, 8, 16)
    for bad in ({"k": k.to("meta")}, {"v": v.to("meta")}, {"rope": torch.zeros(1024, 64, device="meta").bfloat16()}):
        args = {"k": k, "v": v, "rope": None, **bad}
        if dev.type == "cuda" and args["rope"] is None:
            continue                                          # (a tensor that is on no GPU at all has an error of its own)
        with pytest.raises(ValueError, match="one device"):
            llsa_amd.llsa_l1(q, args["k"], args["v"], 8, 16, rope=args["rope"])
    x, (perm, inv) = torch.randn(1, 64, 8, device=dev).requires_grad_(), _permutation(dev)
    y = llsa_amd.permute_tokens(x, perm, None)
    assert torch.equal(y, x[:, perm.long(), :])
    with pytest.raises(ValueError, match="inverse"):
        y.sum().backward()
