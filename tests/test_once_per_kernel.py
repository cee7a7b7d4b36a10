"""What the runtime is asked once per kernel and device (csrc/once_per_kernel.hpp): of every kernel, also where several take the same
arguments, and a refusal is remembered.  Host code, compiled here for the CPU."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncase_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    tmp_path = tmp_path_factory.mktemp("once")
    (tmp_path / "o.cpp").write_text("""#include "once_per_kernel.hpp"
template <int V> void kernel(int) {}
static int asked[3];
template <int V> int ask(int device, int answer) {
    return nnhip::once_per_kernel<kernel<V>>(device, [&] { asked[V]++; return answer; });
}
extern "C" int call(int v, int device, int answer) { return v == 0 ? ask<0>(device, answer) : v == 1 ? ask<1>(device, answer) : ask<2>(device, answer); }
extern "C" int count(int v) { return asked[v]; }
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(tmp_path / "o.cpp"), "-o", str(tmp_path / "o.so"), "-pthread"])
    return C.CDLL(str(tmp_path / "o.so"))


def test_each_kernel_and_device_is_asked_for_once(lib):
    for _ in range(3):
        for v in range(3):
            for device in (0, 1, 15):
                assert lib.call(v, device, 0) == 0
    assert [lib.count(v) for v in range(3)] == [3, 3, 3]


def test_a_refusal_is_told_to_every_later_call(lib):
    assert lib.call(0, 8, 7) == 7
    assert lib.call(0, 8, 0) == 7 and lib.call(1, 8, 0) == 0 and lib.call(0, 9, 0) == 0
