"""The membrane kernels' launch at any number of vertices: a grid the runtime takes (fewer than 2^32
threads), which covers the vertices at 32 lanes each or walks them with a stride."""
import ctypes as C
import os
import subprocess

import pytest

from natray_amd.build import CSRC, HIPCC, ROOT


@pytest.fixture(scope="module")
def groups(tmp_path_factory):
    d = tmp_path_factory.mktemp("groups")
    src, lib = d / "groups.cpp", d / "groups.so"
    src.write_text('#include <hip/hip_runtime.h>\n#include "natray_dev.h"\nextern "C" uint32_t groups(uint32_t g) { return natray::mem_groups(g); }\n')
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", f"-I{CSRC}",
                    f"-I{os.path.join(ROOT, 'include')}", str(src), "-o", str(lib)], check=True)
    fn = C.CDLL(str(lib)).groups
    fn.restype, fn.argtypes = C.c_uint32, [C.c_uint32]
    return fn


@pytest.mark.parametrize("verts", [1, 255, 257, 40962, (1 << 25) - 1, 1 << 25, (1 << 27) - 1, 1 << 27, 1 << 30, (1 << 32) - 256])
def test_grid(groups, verts):
    at_a_thread_each = (verts + 255) // 256
    g = groups(at_a_thread_each)
    assert 1 <= g and g * 256 < 1 << 32
    assert g * 8 >= min(verts, 1 << 25)  # eight vertices a workgroup, each once where they fit
    assert g == min(at_a_thread_each * 32, 1 << 22)
