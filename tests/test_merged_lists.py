"""merge_lists of llsa_device.h, compiled by itself for the CPU: the merged lists of sibling query blocks against sets, with block ids
up to the largest a 32-bit token count allows."""
import ctypes as C
import os
import subprocess

import pytest
import torch

SOURCE = r"""
#include "llsa_device.h"
using namespace llsa;
template <int Q, int R>
__global__ void kernel(const int* ip, int T, int N1, int* out) {
    __shared__ int scratch[R * kWave];
    const int lane = threadIdx.x;
    MergedLists<Q, R> ml = merge_lists<Q, R>(ip, T, N1, lane, scratch);
    for (int i = 0; i < ml.n; i++) {
        const int b = ml.block(i), s = (int)ml.rows(i);
        if (lane == 0) out[1 + 2 * i] = b, out[2 + 2 * i] = s;
    }
    if (lane == 0) out[0] = ml.n;
}
extern "C" void run(int Q, int R, const int* ip, int T, int N1, int* out) {
    if (Q == 1) hipLaunchKernelGGL(HIP_KERNEL_NAME(kernel<1, 1>), dim3(1), dim3(64), 0, nullptr, ip, T, N1, out);
    else if (R == 1) hipLaunchKernelGGL(HIP_KERNEL_NAME(kernel<2, 1>), dim3(1), dim3(64), 0, nullptr, ip, T, N1, out);
    else hipLaunchKernelGGL(HIP_KERNEL_NAME(kernel<2, 2>), dim3(1), dim3(64), 0, nullptr, ip, T, N1, out);
}
"""


@pytest.fixture(scope="module")
def merge(tmp_path_factory):
    from emu_util import emu_lib                              # (with the path of tests/cpu_emu)
    import build_emu
    emu_lib()                                                 # (skips where no host clang can build it)
    d = tmp_path_factory.mktemp("merge")
    (d / "merge.cpp").write_text(SOURCE)
    subprocess.run([build_emu.CLANG, "-std=c++17", "-O1", "-fPIC", "-shared", "-I", os.path.join(build_emu.HERE, "include"), "-I", build_emu.CSRC,
                    "-Wno-everything", "-ffp-contract=off", "-DLLSA_CPU_EMU_BUILD", str(d / "merge.cpp"),
                    os.path.join(build_emu.HERE, "emu_runtime.cpp"), "-o", str(d / "merge.so")], check=True)
    lib = C.CDLL(str(d / "merge.so"))

    def call(rows, N1, R):
        Q, T = rows.shape
        ip, out = rows.int().contiguous(), torch.full((1 + 2 * Q * T,), -1, dtype=torch.int32)
        lib.run(Q, R, C.c_void_p(ip.data_ptr()), T, N1, C.c_void_p(out.data_ptr()))
        n = int(out[0])
        return out[1:1 + 2 * n].reshape(n, 2).tolist()
    return call


@pytest.mark.parametrize("N1", [64, 2 ** 24, 2 ** 24 + 1024, 2 ** 27 - 1])      # 2^27 - 1: beyond N = 2^31 - 16 there is no int32 token count
@pytest.mark.parametrize("Q,R,T", [(1, 1, 64), (2, 1, 4), (2, 1, 32), (2, 2, 48), (2, 2, 64)])
def test_against_sets(merge, Q, R, T, N1):
    g = torch.Generator().manual_seed(T)
    near_end = lambda: N1 - 1 - torch.randperm(64, generator=g)[:T]
    rows = torch.stack([near_end() for _ in range(Q)])
    rows[:, : T // 2] = rows[:1, : T // 2]                    # siblings share blocks
    if Q == 2:
        for i in range(T // 2, T):                            # (and stay distinct within a row)
            while rows[1, i] in rows[1, :i]:
                rows[1, i] = N1 - 1 - torch.randint(0, 64, (1,), generator=g)
    ref = {}
    for u in range(Q):
        for b in rows[u].tolist():
            ref[b] = ref.get(b, 0) | 1 << u
    got = merge(rows, N1, R)
    assert len(got) == len(ref) and {b: s for b, s in got} == ref


@pytest.mark.parametrize("T", [4, 12, 16, 20, 28, 32])        # two lists in either half of a wave: up to sixteen entries, and beyond
@pytest.mark.parametrize("shared", ["none", "all turned", "last with first", "one row repeats its last"])
def test_two_short_lists(merge, T, shared):
    N1 = 4096
    rows = torch.randperm(N1, generator=torch.Generator().manual_seed(T))[: 2 * T].reshape(2, T)
    if shared == "all turned":
        rows[1] = rows[0].roll(T // 2 + 1)
    elif shared == "last with first":
        rows[1, 0] = rows[0, T - 1]
    elif shared == "one row repeats its last":
        rows[1, T - 1] = rows[1, 0]
    got = merge(rows, N1, 1)
    if shared == "one row repeats its last":                  # every entry on its own
        assert sorted(map(tuple, got)) == sorted((int(b), 1 << u) for u in range(2) for b in rows[u])
        return
    ref = {}
    for u in range(2):
        for b in rows[u].tolist():
            ref[b] = ref.get(b, 0) | 1 << u
    assert len(got) == len(ref) and {b: s for b, s in got} == ref
    assert [s for _, s in got] == sorted((s for _, s in got), reverse=True)
