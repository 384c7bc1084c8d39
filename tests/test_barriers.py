"""Work-group barriers and exchanges within a wave, read from the sources: a
device function that a kernel calls from a branch on the wave holds no
work-group barrier (the language promises nothing when a work-group's waves meet
at different ones), and lanes hand LDS values to each other only past a fence
(__builtin_amdgcn_wave_barrier alone orders nothing in memory)."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mast-multiphysics_amd", "csrc")


def _text(f):
    return re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, f)).read())


def _body(text, name):
    m = re.search(r"\b%s\([^;{}]*\)\s*\{" % name, text)
    depth, i = 1, m.end()
    while depth:
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        i += 1
    return text[m.end():i - 1]


def test_no_work_group_barrier_in_a_branch_on_the_wave():
    text = _text("mg_kernels.hip")
    assert re.search(r"if \(layer == 0\) stencil_layer<0>", text)
    assert "__syncthreads" not in _body(text, "stencil_layer")


def test_exchanges_within_a_wave_are_fenced():
    for f in sorted(os.listdir(CSRC)):
        text = _text(f)
        if f == "device_util.h":
            body = _body(text, "wave_exchange")
            assert body.count("__builtin_amdgcn_fence") == 2
            assert body.index("__ATOMIC_RELEASE") < body.index("wave_barrier") < body.index("__ATOMIC_ACQUIRE")
            text = text.replace(body, "")
        assert "__builtin_amdgcn_wave_barrier" not in text, f
