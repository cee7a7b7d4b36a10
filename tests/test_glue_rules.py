"""The turns a pooling window is taken in (csrc/glue_rules.hpp, compiled here for the CPU): no more of them than five values a turn
need, and fewer values asked for past the window's end than there are turns."""
import ctypes as C
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncase_amd", "csrc")


def test_a_window_is_spread_evenly_over_its_turns(tmp_path):
    (tmp_path / "r.cpp").write_text('#include "glue_rules.hpp"\nextern "C" int loads(int window) { return nnhip::loads_per_turn(window); }\n')
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(tmp_path / "r.cpp"), "-o", str(tmp_path / "r.so")])
    loads = C.CDLL(str(tmp_path / "r.so")).loads
    for window in range(1, 64):
        turns = -(-window // loads(window))
        assert 1 <= loads(window) <= 5 and turns == -(-window // 5)
        assert turns * loads(window) - window < turns
