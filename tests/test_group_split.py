"""The group-major pass where the groups of its last round are dealt out to several workgroups, against the oracle.  An XCD has 8 groups per head of
16384 tokens and takes 64 at a time: 1, 4 and 7 heads are one round that is an eighth, half and seven eighths full, 8 fill it, 9, 10 and 12 leave a
second one nearly empty to half full; few key blocks a group (T2 + 4) are dealt out to fewer workgroups or none, many to more waves than
have a share."""
import ctypes as C
import os
import subprocess

import pytest
import torch

import parity_cases as P


def test_no_workgroup_without_key_blocks(tmp_path):
    """The split itself, compiled from the kernel's source: its parts are as many workgroups as find room in the last round, and every one has key blocks."""
    from emu_util import emu_lib                              # (with the path of tests/cpu_emu)
    import build_emu
    emu = emu_lib().path
    (tmp_path / "split.cpp").write_text('''
#include "attn_bwd.hip"
extern "C" void split(int groups, int n_blocks, int* out) {
    const GroupSplit s = group_split(groups, n_blocks);
    out[0] = s.whole, out[1] = s.parts, out[2] = kGroupSlots, out[3] = kGroupWaves;
}
''')
    subprocess.run([build_emu.CLANG, "-std=c++17", "-O0", "-fPIC", "-shared", "-I", os.path.join(build_emu.HERE, "include"), "-I", build_emu.CSRC,
                    "-Wno-everything", "-ffp-contract=off", "-DLLSA_CPU_EMU_BUILD", str(tmp_path / "split.cpp"), emu, "-o", str(tmp_path / "split.so")], check=True)
    lib, out, dealt = C.CDLL(str(tmp_path / "split.so")), (C.c_int * 4)(), 0
    for rounds in (0, 2):
        for rest in range(64):
            for n_blocks in range(8, 65):
                lib.split(64 * rounds + rest, n_blocks, out)
                whole, parts, slots, waves = out
                assert slots == 64 and parts >= 1 and (rest or parts == 1)
                if parts == 1:
                    assert whole == 64 * rounds + rest
                    continue
                dealt += 1
                per = -(-n_blocks // (waves * parts))         # key blocks a wave has at most, as the kernel deals them
                assert whole == 64 * rounds and rest * parts <= slots
                assert (parts - 1) * waves * per < n_blocks, (rest, n_blocks, parts)
    assert dealt > 1000


@pytest.mark.gpu
@pytest.mark.parametrize("H,T2", [(1, 4), (1, 8), (1, 16), (1, 32), (4, 16), (7, 16), (8, 16), (9, 4), (9, 8), (9, 20), (9, 32), (10, 16), (12, 24)])
def test_grids(H, T2):
    P.check_op_l2(torch.device("cuda"), B=1, H=H, N=16384, T=8, T2=T2, fused=True, rope=True, smooth=True)
