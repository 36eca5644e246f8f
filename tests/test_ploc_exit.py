"""The clustering's early exit (internal.h, built here for the host): whatever the waves of a launch read
of the word that the same launch sets, they take the same way. No GPU."""
import ctypes
import subprocess

import pytest

import portablert_amd.build as build

SRC = """
#include "internal.h"
extern "C" unsigned held_by(unsigned step) { return prt::held_by(step); }
extern "C" int held_before(unsigned held, unsigned step) { return prt::held_before(held, step); }
extern "C" unsigned held_buffer(unsigned held) { return prt::held_buffer(held); }
"""


@pytest.fixture(scope="module")
def held(tmp_path_factory):
    d = tmp_path_factory.mktemp("held")
    src, so = d / "held.hip", d / "held.so"
    src.write_text(SRC)
    subprocess.run([build.HIPCC, "--offload-host-only", "-std=c++17", "-O2", "-fPIC", "-shared",
                    "-I" + build.CSRC, str(src), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def test_waves_of_a_launch_agree(held):
    steps = 40
    for found in range(1, steps):  # the step that finds few enough clusters
        word = 0
        for step in range(1, steps):
            before = bool(held.held_before(word, step))
            written = held.held_by(step) if step >= found and not before else word
            # a wave reads the word as the launch found it or as the launch's first workgroup left it
            assert {bool(held.held_before(w, step)) for w in (word, written)} == {before}
            assert before == (step > found)
            word = written
        assert held.held_buffer(word) == found & 1
