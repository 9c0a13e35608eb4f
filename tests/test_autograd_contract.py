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
