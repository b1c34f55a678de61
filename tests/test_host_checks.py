"""CPU: the Python bindings check buffer sizes and shapes before they hand raw
pointers to the library (no device call is reached on these paths)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import bec_amd as B
from bec_amd import fno as F


def _fake_device_array(nbytes):
    d = F.DeviceArray.__new__(F.DeviceArray)
    d.shape, d.dtype, d.nbytes = (nbytes // 4,), np.dtype(np.float32), nbytes
    d.ptr = C.c_void_p(0x10000)
    return d


def _calc():
    return B.derive(B.default_model(N=30000, nvx=16, nvy=16, nvz=128, ne=1))


def test_gs2_features_rejects_short_buffer():
    c = _calc()
    short = _fake_device_array(c.cells * 64 - 4)
    with pytest.raises(ValueError, match="need"):
        F.gs2_features(c, [0.0, 0.0, 0.0, 0.0], short)
    # a view that starts inside the allocation has only the rest of it
    base = _fake_device_array(2 * c.cells * 64)
    view = F.DeviceView(base, c.cells * 64 + 4)
    with pytest.raises(ValueError, match="need"):
        F.gs2_features(c, [0.0, 0.0, 0.0, 0.0], view)
    with pytest.raises(ValueError):
        F.gs2_features(c, [0.0, 0.0, 0.0], _fake_device_array(c.cells * 64))
    short.ptr = base.ptr = C.c_void_p()   # nothing to free


def test_set_state_rejects_wrong_shape():
    s = B.Solver.__new__(B.Solver)
    s.groups = [_calc()]
    s._ctx = C.c_void_p()
    good = np.zeros(s.shape(0), dtype=complex)
    with pytest.raises(ValueError, match="shape"):
        s.set_state(good[:, :8], good)
    with pytest.raises(ValueError, match="shape"):
        s.set_state(good, good.reshape(-1))


HARNESS_PLACE = r"""
#include <stdio.h>
#include "output_place.hpp"
int main() {
    unsigned long long v[9];
    while (fread(v, sizeof(v), 1, stdin) == 1) {
        bec::OutputPlace p;
        p.device_memory = v[0] != 0;
        p.device = (int)v[1];
        p.base = v[2];
        p.size = v[3];
        putchar(bec::writes_direct(p, (int)v[4], v[5], v[6], v[7], v[8]) ? '1' : '0');
    }
    return 0;
}
"""


def test_only_own_device_memory_apart_from_the_input_is_written_directly(tmp_path):
    """Where the network's last kernel stores straight into the caller's output: memory of another device
    (no kernel may reach it without peer access), host memory and outputs that overlap the input are copied."""
    src, exe = tmp_path / "h.cpp", tmp_path / "h"
    src.write_text(HARNESS_PLACE)
    subprocess.run(["g++", "-O2", "-I", os.path.join(os.path.dirname(B.__file__), "csrc"), str(src), "-o", str(exe)],
                   check=True)
    base, size, x = 0x1000000, 4096, 0x2000000
    top = 2 ** 64 - 4096
    cases = [   # device memory, its device, allocation, size, own device, output, bytes, input, bytes
        ((1, 0, base, size, 0, base, size, x, 4096), 1),
        ((1, 3, base, size, 3, base + 96, size - 96, x, 4096), 1),
        ((1, 1, base, size, 0, base, size, x, 4096), 0),             # another device's
        ((0, 0, base, size, 0, base, size, x, 4096), 0),             # host memory
        ((1, 0, base, size, 0, base, size + 4, x, 4096), 0),         # larger than the allocation
        ((1, 0, base, size, 0, base + 4, size, x, 4096), 0),
        ((1, 0, base, size, 0, base + 2, 64, x, 4096), 0),           # not a float's address
        ((1, 0, base, size, 0, base - 4, 64, x, 4096), 0),
        ((1, 0, base, size, 0, base + size + 4, 4, x, 4096), 0),
        ((1, 0, base, size, 0, base, 2 ** 64 - 4, x, 4096), 0),      # no sum overflows
        ((1, 0, top, 4096, 0, top + 64, 2 ** 63, x, 4096), 0),
        ((1, 0, base, size, 0, base + 2048, 1024, base, 2048), 1),   # behind the input, before it
        ((1, 0, base, size, 0, base, 1024, base + 1024, 2048), 1),
        ((1, 0, base, size, 0, base + 2044, 1024, base, 2048), 0),   # over its end, its start, inside, around, the same
        ((1, 0, base, size, 0, base, 1028, base + 1024, 2048), 0),
        ((1, 0, base, size, 0, base + 64, 64, base, 2048), 0),
        ((1, 0, base, size, 0, base, 4096, base + 64, 64), 0),
        ((1, 0, base, size, 0, base, 1024, base, 2048), 0),
    ]
    data = np.array([c for c, _ in cases], dtype=np.uint64)
    out = subprocess.run([str(exe)], input=data.tobytes(), stdout=subprocess.PIPE, check=True).stdout.decode()
    assert out == "".join(str(w) for _, w in cases)
