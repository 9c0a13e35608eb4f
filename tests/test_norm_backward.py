"""The backward of the qk RMS norm inside the kernels that write dq and dk: the operator with the norm against the same
operator on rows normalised beforehand, its dq and dk taken back through the norm in fp32.  Sizes: one and two query blocks
per wave, one and two list registers, a key block whose queries are one piece and one cut into several."""
import pytest
import torch

import parity_cases as P
from llsa_amd.kernel.hip.rms_norm import rms_norm_fwd
from llsa_amd.kernel.torch_op.flash_sparse_attention_res_1 import llsa_l1

pytestmark = pytest.mark.gpu


def _reference(dy, x, gamma, eps):
    dy, x, gamma = dy.double(), x.double(), gamma.double()
    rstd = (x.square().mean(-1, keepdim=True) + eps).rsqrt()
    xn, g = x * rstd, dy * gamma
    return rstd * (g - xn * (g * xn).mean(-1, keepdim=True)), (dy * xn).sum((0, 1, 2))


@pytest.mark.parametrize("B,H,N,T,rope,smooth,aligned", [(1, 1, 1024, 8, True, False, True), (1, 3, 1024, 64, False, True, False),
                                                         (1, 64, 1024, 8, True, True, True), (4, 4, 4096, 36, False, False, True)])
def test_against_the_operator_without_norm(B, H, N, T, rope, smooth, aligned):
    from llsa_amd.utils.rope_table import rope_table
    dev = torch.device("cuda")
    q, k, v, do = P.smooth_inputs(B, H, N, 64, dev) if smooth else P.randn_inputs(B, H, N, 64, dev, seed=19, strided=True)
    freq = rope_table(int(N ** 0.5), dtype=torch.bfloat16).to(dev) if rope else None
    gq, gk, eps = P._norm_weights(dev)
    if not aligned:                                           # weights on 4-byte boundaries
        gq, gk = (torch.cat([g[:1], g])[1:] for g in (gq, gk))
    gq.requires_grad_(), gk.requires_grad_()
    a = [t.detach().clone().requires_grad_() for t in (q, k, v)]
    llsa_l1(*a, T, 16, rope=freq, qk_norm=(gq, gk, eps)).backward(do)
    b = [t.detach().requires_grad_() for t in (rms_norm_fwd(q, gq.detach(), eps), rms_norm_fwd(k, gk.detach(), eps), v)]
    llsa_l1(*b, T, 16, rope=freq).backward(do)
    for name, got, dgot, dy, x, gamma in (("q", a[0].grad, gq.grad, b[0].grad, q, gq), ("k", a[1].grad, gk.grad, b[1].grad, k, gk)):
        dx, dg = _reference(dy, x, gamma.detach(), eps)
        err = (got.double() - dx).abs() / (2.0 ** -8 * dx.abs() + 1e-4 * dx.abs().max())
        assert err.max() < 1.1, (name, float(err.max()))      # bf16 rounding of the result
        assert (dgot - dg).abs().max() <= 1e-4 * dg.abs().max() + 1e-4, name
    assert torch.equal(a[2].grad, b[2].grad)
