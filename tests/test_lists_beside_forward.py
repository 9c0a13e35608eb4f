"""The index transposes made by workgroups of the forward attention launch: the same lists, and the same output, as in launches of
their own -- one range and many, rows that do not divide, repeated entries, grids of one and of two query blocks a wave, and lists too long or
too many to ride along."""
import ctypes as C
import os
import subprocess

import pytest
import torch

import parity_cases as P
from emu_util import emu_lib
from llsa_amd._lib import TransposeJob, current_lib, override_library_for_tests


def _check(dev, monkeypatch, B, H, N, T, T2, chunk):
    from llsa_amd.kernel.hip._attention import attn_fwd
    from llsa_amd.kernel.hip.indices_transpose import transpose_indices_levels
    from llsa_amd.kernel.hip.mean_pool import mean_pool1d
    lib = current_lib()
    q, k, v, _ = P.randn_inputs(B, H, N, 64, dev, seed=N + T)
    pk, pv = mean_pool1d(k, 16), mean_pool1d(v, 16)
    sels = [P._hot_indices(B, H, N // 16, N // 16, T, 3, 11).int().to(dev)]
    kw = {}
    if T2:
        sels.append(P._hot_indices(B, H, N // 256, N // 256, T2, 1, 12).int().to(dev))
        kw = {"pk2": mean_pool1d(pk, 16), "pv2": mean_pool1d(pv, 16), "p_indices": sels[1], "token_weight_2": 256.0}
    sels[0][:, :, 5, 1] = sels[0][:, :, 5, 0]                 # a repeated entry
    o, lse = attn_fwd(q, k, v, pk, pv, sels[0], 16.0, **kw)
    ref = transpose_indices_levels(sels, chunk)
    got = [tuple(torch.full_like(t, -7) for t in r) for r in ref]
    jobs = (TransposeJob * len(sels))()
    for l, (sel, (off, flat, extra)) in enumerate(zip(sels, got)):
        Mb, Ts = sel.shape[2:]
        jobs[l] = TransposeJob(sel.data_ptr(), off.data_ptr(), flat.data_ptr(), None if l else extra.data_ptr(), extra.data_ptr() if l else None,
                               Mb, Mb, Ts, 1 if l else chunk)
    monkeypatch.setattr(lib, "attn_fwd", lambda a, stream: lib.attn_fwd_lists(a, jobs, len(sels), stream))
    o2, lse2 = attn_fwd(q, k, v, pk, pv, sels[0], 16.0, **kw)
    monkeypatch.undo()
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    for l, (a, b) in enumerate(zip(ref, got)):
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]), f"level {l + 1}"
        if l:
            assert torch.equal(a[2], b[2])
            continue
        multi = 4 + 4 * (N // 16 * T // chunk + N // 16)      # where the records of the cut lists begin
        for x, y in zip(a[2].reshape(-1, a[2].shape[-1]).cpu(), b[2].reshape(-1, b[2].shape[-1]).cpu()):
            items, cut = int(x[0]), int(x[2])
            assert torch.equal(x[:4 + 4 * items], y[:4 + 4 * items]) and torch.equal(x[multi:multi + 4 * cut], y[multi:multi + 4 * cut])


@pytest.mark.parametrize("B,H,N,T,T2,chunk", [(1, 2, 1024, 4, 0, 16), (1, 1, 2048, 12, 0, 32)])
def test_cpu(monkeypatch, B, H, N, T, T2, chunk):
    with override_library_for_tests(emu_lib()):
        _check(torch.device("cpu"), monkeypatch, B, H, N, T, T2, chunk)


def _ride(B, H, N, *topk):
    return current_lib().lists_ride(B, H, N, (C.c_int32 * len(topk))(*topk), len(topk))


def test_lines_of_the_rule():
    assert _ride(1, 6, 1024, 8) and _ride(2, 6, 16384, 16, 16) and _ride(1, 6, 65536, 16, 16) and _ride(3, 5, 7168, 12)
    assert _ride(1, 20, 65536, 16, 16) and not _ride(1, 24, 65536, 16, 16) and not _ride(1, 32, 65536, 16, 16)    # entries read: 88, 105 and 141 million
    assert _ride(16, 8, 16384, 64, 16) and _ride(128, 16, 1024, 8)
    assert not _ride(1, 1, 65536, 20, 8)                      # more than 65536 entries
    assert _ride(1, 1, 130048, 8) and not _ride(1, 1, 131072, 8, 4)      # 8128 and 8192 key blocks: their histogram takes 8160 ints of LDS at most
    assert not _ride(1, 65535, 1024, 4)                       # more rows than a grid has


def test_the_query_plans_the_operators_jobs(tmp_path):
    """llsa_lists_ride asks for the plan of the jobs that the operators pass: inverse positions, which double a key block's LDS, of every level but the first."""
    emu = emu_lib().path                                      # (with the path of tests/cpu_emu)
    import build_emu
    (tmp_path / "ride.cpp").write_text('''
#include "attn_fwd.hip"
static int seen[LLSA_MAX_LEVELS];
bool llsa::plan_transpose(const llsa_transpose_job* jobs, int n_jobs, int, int, int, TrJobs& plan) {
    for (int i = 0; i < n_jobs; i++) seen[i] = jobs[i].inv != nullptr ? 2 : 1;
    plan = TrJobs{};
    return true;
}
extern "C" int ride(int N, const int32_t* topk, int levels, int* out) {
    const int rc = llsa_lists_ride(1, 1, N, topk, levels);
    for (int i = 0; i < levels; i++) out[i] = seen[i];
    return rc;
}
''')
    subprocess.run([build_emu.CLANG, "-std=c++17", "-O0", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-I", os.path.join(build_emu.HERE, "include"), "-I",
                    build_emu.CSRC, "-Wno-everything", "-ffp-contract=off", "-DLLSA_CPU_EMU_BUILD", str(tmp_path / "ride.cpp"), emu, "-o",
                    str(tmp_path / "ride.so")], check=True)
    lib = C.CDLL(str(tmp_path / "ride.so"))
    for levels, N in ((1, 1024), (2, 16384), (3, 262144)):
        out = (C.c_int * levels)()
        assert lib.ride(N, (C.c_int32 * levels)(*[8] * levels), levels, out) == 1
        assert list(out) == [1] + [2] * (levels - 1)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,T,T2,chunk", [(1, 24, 4096, 4, 0, 64), (1, 16, 16384, 48, 4, 64)])
def test_two_query_blocks_a_wave(monkeypatch, B, H, N, T, T2, chunk):
    topk = (T, T2) if T2 else (T,)
    assert current_lib().query_blocks_per_wave(B, H, N, (C.c_int32 * len(topk))(*topk), len(topk), 0) == 2 and _ride(B, H, N, *topk)
    _check(torch.device("cuda"), monkeypatch, B, H, N, T, T2, chunk)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,T,T2,chunk", [(1, 1, 131072, 8, 4, 256), (1, 24, 65536, 16, 4, 256)])
def test_behind_the_forward(monkeypatch, B, H, N, T, T2, chunk):
    """Lists that one launch could make, but not beside the attention: too many key blocks, too many entries over all heads."""
    topk = (C.c_int32 * 2)(T, T2)
    assert current_lib().transpose_one_launch(N // 16, N // 16, T, B, H) and not current_lib().lists_ride(B, H, N, topk, 2)
    _check(torch.device("cuda"), monkeypatch, B, H, N, T, T2, chunk)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,T,T2,chunk", [(1, 2, 1024, 4, 0, 16), (3, 5, 7168, 12, 0, 64), (1, 1, 4096, 64, 0, 64), (2, 6, 16384, 16, 16, 64),
                                              (1, 1, 65536, 16, 4, 256), (1, 1, 32768, 32, 8, 256), (1, 1, 65536, 20, 8, 256), (1, 1, 49152, 64, 32, 256)])
def test_gpu(monkeypatch, B, H, N, T, T2, chunk):
    _check(torch.device("cuda"), monkeypatch, B, H, N, T, T2, chunk)
