"""How the wide prompt pass shares tiles out that are no multiple of the compute units (TileShare in slai_amd/csrc/wide_layout.h), walked on the CPU."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("share") / "libtile_share.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-I", os.path.join(ROOT, "slai_amd", "csrc"), os.path.join(HERE, "native", "tile_share.cpp"), "-o", out])
    L = C.CDLL(out)
    L.share_walk.argtypes = [C.c_uint32] * 3 + [C.POINTER(C.c_uint32), C.c_char_p, C.c_size_t]

    def run(units, blocks, ncb):
        longest, msg = C.c_uint32(), C.create_string_buffer(200)
        return L.share_walk(units, blocks, ncb, C.byref(longest), msg, 200), msg.value.decode(), longest.value
    return run


@pytest.mark.parametrize("units", [1, 7, 8, 9, 24, 43, 74, 150])
@pytest.mark.parametrize("ncb", [1, 2, 3, 14, 16, 43])
def test_every_super_block_once(walk, units, ncb):
    for blocks in range(1, 17):
        rc, msg, longest = walk(units, blocks, ncb)
        assert rc == 0, (blocks, msg)
        per_die = -(-units * blocks // 8)
        assert per_die * ncb <= 32 * longest <= 32 * ncb * -(-per_die // 32)      # no less than an even share, no more than whole rounds
