"""The table that the four lanes of a quad share (csrc/kern_quad.hpp): one lane writes it and all read it,
so secp_build_table has to order the writes before the other lanes' reads, and those reads before the
next writes to the same words. The host build runs it under that memory model."""
import ctypes
import os
import subprocess

import pytest

import pyref

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "wgpu-sigops_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("quad_table") / "libquad_table.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-DSIGOPS_HOST_CHECK=1",
                    "-I" + CSRC, "-o", so, os.path.join(HERE, "devcheck", "quad_table_check.cpp")], check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("curve", [0, 1])
def test_shared_table_is_ordered(lib, curve):
    c = pyref.CURVES[curve]
    for k in (1, 2, 3, 0x1234567):
        P = pyref.w_mul(c, c["G"], k)
        assert lib.qt_check(curve, P[0].to_bytes(32, "big") + P[1].to_bytes(32, "big")) == 0
