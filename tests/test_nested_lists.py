"""The transposed lists of a selection that is nested in the one above it, made from that one's lists: the same offsets, segments and work
list as from the general form -- numbers of owners and parents that do not fill a workgroup, one to 64 parents, lists cut into pieces,
segments without an entry."""
import pytest
import torch

from emu_util import emu_lib
from llsa_amd._lib import TransposeJob, current_lib, override_library_for_tests
from llsa_amd.kernel.hip._common import stream_of


def _nested(BH, owners, parents, T, Tp, seed):
    """(BH, owners, Tp) parents, some of them popular, and (BH, 16 owners, T) children of those"""
    g = torch.Generator().manual_seed(seed)
    weight = torch.rand(BH, owners, parents, generator=g) + 2.0 * (torch.arange(parents) < max(1, parents // 8))
    top = weight.topk(Tp, -1).indices
    cand = (top[..., None] * 16 + torch.arange(16)).reshape(BH, owners, 1, Tp * 16).expand(-1, -1, 16, -1)
    pick = (torch.rand(BH, owners, 16, Tp * 16, generator=g) + 1.0 * (cand % 16 == 3)).topk(T, -1).indices
    return top.int(), cand.gather(-1, pick).reshape(BH, owners * 16, T).int()


def _check(dev, BH, owners, parents, T, Tp, chunk):
    lib = current_lib()
    top, sel = (t.contiguous().to(dev) for t in _nested(BH, owners, parents, T, Tp, owners + T))
    Mb, Kb = owners * 16, parents * 16
    wl = lib.work_list_len(Mb, Kb, T, chunk)
    out = []
    for nested in (False, True):
        buf = dict(off=torch.full((BH, Kb + 1), -7), flat=torch.full((BH, Mb * T), -7), work=torch.full((BH, wl), -7),
                   p_off=torch.full((BH, parents + 1), -7), p_flat=torch.full((BH, owners * Tp), -7), p_inv=torch.full((BH, owners, Tp), -7))
        buf = {k: v.int().to(dev) for k, v in buf.items()}
        scratch = torch.full((lib.transpose_nested_bytes(Mb, Kb, Tp, 1, BH),), 0xA5, dtype=torch.uint8).to(dev)
        jobs = (TransposeJob * 2)(
            TransposeJob(sel.data_ptr(), buf["off"].data_ptr(), buf["flat"].data_ptr(), buf["work"].data_ptr(), None, Mb, Kb, T, chunk,
                         scratch.data_ptr() if nested else None),
            TransposeJob(top.data_ptr(), buf["p_off"].data_ptr(), buf["p_flat"].data_ptr(), None, buf["p_inv"].data_ptr(), owners, parents, Tp, 1))
        lib.check(lib.transpose_indices_multi(jobs, 2, 1, BH, stream_of(lib, sel)), "transpose_indices")
        out.append({k: v.cpu() for k, v in buf.items()})
    a, b = out
    for k in ("off", "flat", "p_off", "p_flat", "p_inv"):
        assert torch.equal(a[k], b[k]), k
    multi = 4 + 4 * (Mb * T // chunk + Kb)
    cuts = 0
    for x, y in zip(a["work"], b["work"]):
        assert torch.equal(x[:4], y[:4])
        items, cut = int(x[0]), int(x[2])
        assert torch.equal(x[4:4 + 4 * items], y[4:4 + 4 * items]) and torch.equal(x[multi:multi + 4 * cut], y[multi:multi + 4 * cut])
        cuts += cut
    return cuts


@pytest.mark.parametrize("BH,owners,parents,T,Tp,chunk", [(2, 5, 19, 4, 1, 4), (1, 9, 33, 20, 4, 8), (1, 4, 64, 64, 64, 16)])
def test_cpu(BH, owners, parents, T, Tp, chunk):
    with override_library_for_tests(emu_lib()):
        assert _check(torch.device("cpu"), BH, owners, parents, T, Tp, chunk) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("BH,owners,parents,T,Tp,chunk", [(2, 5, 19, 4, 1, 4), (1, 9, 33, 20, 4, 8), (1, 4, 64, 64, 64, 16), (3, 192, 192, 64, 32, 256),
                                                          (2, 1024, 1024, 16, 16, 256), (1, 2048, 2048, 8, 8, 256)])
def test_gpu(BH, owners, parents, T, Tp, chunk):
    _check(torch.device("cuda"), BH, owners, parents, T, Tp, chunk)


def test_wrong_jobs_are_errors():
    with override_library_for_tests(emu_lib()):
        lib = current_lib()
        t = torch.zeros(4096, dtype=torch.int32)
        p = t.data_ptr()
        above = TransposeJob(p, p, p, None, p, 2, 2, 2, 1)
        assert lib.transpose_nested_bytes(32, 32, 65, 1, 1) < 0 and lib.transpose_nested_bytes(40, 32, 4, 1, 1) < 0
        for job, n in ((TransposeJob(p, p, p, None, None, 32, 32, 4, 1, p), 1),            # no job above
                       (TransposeJob(p, p, p, None, p, 32, 32, 4, 1, p), 2),               # asks for its inverse
                       (TransposeJob(p, p, p, None, None, 48, 32, 4, 1, p), 2),            # not the parents' shape
                       (TransposeJob(p, p, p, None, None, 32, 32, 2, 1, p), 2)):           # entries not in fours
            assert lib.transpose_indices_multi((TransposeJob * 2)(job, above), n, 1, 1, None) != 0
