"""Rules that pick a kernel by sizes, compiled for the CPU, at sizes where both
sides were measured."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "asuna_amd", "csrc")
PER_RAY, PACKET, COARSE = 0, 1, 2


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text('#include "device/render.h"\n'
                             'extern "C" int walkOf(uint32_t tris, uint64_t paths, uint64_t pixels, uint64_t views) {\n'
                             '  return int(ashd::cameraWalk(tris, paths, pixels, views));\n}\n')
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC,
                    "-o", str(d / "r.so"), str(d / "r.cpp")], check=True)
    L = C.CDLL(str(d / "r.so"))
    L.walkOf.argtypes = [C.c_uint32, C.c_uint64, C.c_uint64, C.c_uint64]
    return L


@pytest.mark.parametrize("tris,w,h,views,frames,walk", [
    # a tree every wave walks whole, and 8 frames or more of any
    (36, 96, 64, 1, 1, COARSE), (512, 1920, 1080, 1, 1, COARSE), (20_000, 160, 120, 1, 8, COARSE),
    (5_242_880, 1920, 1080, 1, 8, PACKET), (65_537, 64, 64, 1, 9, PACKET),
    # few rays
    (732, 96, 64, 1, 1, PER_RAY), (1_260, 512, 512, 1, 1, PER_RAY), (81_926, 160, 120, 1, 4, PER_RAY),
    # triangles per wave's share of a view: few (732 at 512 x 512: 10 % between the walks), and many
    (732, 512, 512, 1, 2, COARSE), (2_460, 512, 512, 1, 2, COARSE), (5_126, 1920, 1080, 1, 7, COARSE),
    (14_724, 1920, 1080, 1, 4, COARSE), (81_926, 1280, 720, 1, 1, PACKET), (327_686, 1920, 1080, 1, 2, PACKET),
    (14_724, 512, 512, 1, 4, PER_RAY), (24_330, 512, 512, 1, 7, PER_RAY), (327_686, 512, 512, 1, 2, PER_RAY),
    (5_242_880, 1920, 1080, 1, 1, PER_RAY), (5_242_880, 1920, 1080, 1, 4, PER_RAY),
    # a batch of several views counts each view's own paths
    (14_724, 256, 256, 10, 4, PER_RAY), (5_768, 256, 256, 10, 2, PER_RAY), (2_564, 256, 256, 10, 1, PER_RAY),
])
def test_camera_walk_where_both_were_measured(rules, tris, w, h, views, frames, walk):
    assert rules.walkOf(tris, w * h * views * frames, w * h * views, views) == walk


def test_camera_walk_holds_at_any_size(rules):
    big = (1 << 30, 1 << 30, 65535)  # paths, pixels, views of the largest batch
    assert rules.walkOf(0xFFFFFFFF, *big) == PER_RAY
    assert rules.walkOf(0xFFFFFFFF, (1 << 33) - 1, 1 << 30, 1 << 20) == PER_RAY  # products stay in 64 bits
    assert rules.walkOf(0, 0, 0, 0) == COARSE and rules.walkOf(600, 1, 1, 1) == PER_RAY
