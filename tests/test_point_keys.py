"""Layout of the point keys (fwn_order.h, compiled for the host): what the sorts' digits hold."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "o.cpp").write_text('#include "fwn_order.h"\nextern "C" void keys(const uint32_t* c, long n, uint32_t mesh, int bits,'
                             ' int few, uint32_t* k)\n{\n    const int first = few ? 0 : fwn::sort24_first(bits);\n'
                             '    for (long i = 0; i < n; ++i) k[i] = fwn::point_key_of(c[i], mesh, bits, first);\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "lagrange_amd", "csrc"),
                    str(d / "o.cpp"), "-o", str(d / "o.so")], check=True)
    return C.CDLL(str(d / "o.so"))


def keys(lib, code, mesh, bits, few):
    code = np.ascontiguousarray(code, np.uint32)
    k = np.empty_like(code)
    lib.keys(code.ctypes.data_as(C.c_void_p), C.c_long(code.size), C.c_uint32(mesh), bits, int(few),
             k.ctypes.data_as(C.c_void_p))
    return k


@pytest.mark.parametrize("bits", range(9))
def test_sort_of_20_bits(lib, bits):
    """Bits 12 to 31: the mesh, then the 20 - mesh_bits leading bits of the Morton code."""
    code = np.random.default_rng(bits).integers(0, 1 << 30, 10000).astype(np.uint32)
    mesh = (1 << bits) - 1
    want = (code >> (30 - (20 - bits))) | (mesh << (20 - bits))
    np.testing.assert_array_equal(keys(lib, code, mesh, bits, True) >> 12, want)


@pytest.mark.parametrize("bits", [0, 1, 2, 3, 8, 24])
def test_sort_of_24_bits(lib, bits):
    """Bits 8 to 31: the mesh, then 22 leading bits of the Morton code or as many as there is room for; a
    single mesh's keys are the codes."""
    code = np.random.default_rng(bits).integers(0, 1 << 30, 10000).astype(np.uint32)
    mesh = (1 << bits) - 1
    k = keys(lib, code, mesh, bits, False)
    n = min(22, 24 - bits)
    np.testing.assert_array_equal((k >> 8) & ((1 << n) - 1), code >> (30 - n))
    np.testing.assert_array_equal(k >> (32 - bits) if bits else k >> 30, mesh)
    if bits == 0:
        np.testing.assert_array_equal(k, code)
