"""Rows of o, dq, dk and dv that are 8- but not 16-byte aligned: the same values as in aligned rows, and nothing written beside them."""
import ctypes as C

import pytest
import torch

import parity_cases as P
from emu_util import emu_lib
from llsa_amd._lib import current_lib, override_library_for_tests


def _check(dev, monkeypatch, H, N, T):
    from llsa_amd.kernel.hip._attention import attn_bwd, attn_fwd
    from llsa_amd.kernel.hip.mean_pool import mean_pool1d
    lib = current_lib()
    q, k, v, do = P.randn_inputs(1, H, N, 64, dev, seed=N + T)
    pk, pv = mean_pool1d(k, 16), mean_pool1d(v, 16)
    sel = P._hot_indices(1, H, N // 16, N // 16, T, 3, 11).int().to(dev)
    rows = {n: torch.full((1, H, N, 68), 7.0, device=dev, dtype=torch.bfloat16) for n in ("o", "dq", "dk", "dv")}
    fwd, bwd = lib.attn_fwd, lib.attn_bwd

    def moved(call, names):
        def run(a, stream):
            for n in names:
                st = rows[n].stride()
                setattr(a._obj, n, rows[n].data_ptr())
                for axis, s in zip("bhn", st):
                    setattr(a._obj, f"s{n}{axis}", s)
            return call(a, stream)
        return run

    o, lse = attn_fwd(q, k, v, pk, pv, sel, 16.0)
    grads = attn_bwd(do, q, k, v, pk, pv, o, lse, sel, 16.0, 1.0)[:3]
    monkeypatch.setattr(lib, "attn_fwd", moved(fwd, ["o"]))
    monkeypatch.setattr(lib, "attn_bwd", moved(bwd, ["dq", "dk", "dv"]))
    attn_fwd(q, k, v, pk, pv, sel, 16.0)
    attn_bwd(do, q, k, v, pk, pv, o, lse, sel, 16.0, 1.0)
    monkeypatch.undo()
    for n, ref in zip(rows, (o, *grads)):
        assert torch.equal(rows[n][..., :64], ref), n
        assert (rows[n][..., 64:] == 7).all(), n


def test_cpu(monkeypatch):
    with override_library_for_tests(emu_lib()):
        _check(torch.device("cpu"), monkeypatch, 1, 1024, 4)


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,T", [(2, 1024, 8), (24, 4096, 16)])
def test_gpu(monkeypatch, H, N, T):
    _check(torch.device("cuda"), monkeypatch, H, N, T)
