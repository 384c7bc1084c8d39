"""The Krylov kernels hand the solver's scalars from launch to launch, and every
work-group of a launch reads them for itself: a launch of several work-groups
that wrote one of the scalars it reads would race with itself (a work-group that
starts late sees the new value, wave by wave).  Read from the sources: no such
kernel reads a member of CGScalars / BiCGScalars that it writes."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mast-multiphysics_amd", "csrc")
FILES = ["kernels.hip", "mg_kernels.hip", "lattice_box.hip", "mg_tail.hip", "device_util.h"]


def _functions():
    """name -> (is a kernel, body) of every device function of the files."""
    out = {}
    for f in FILES:
        text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, f)).read())
        text = re.sub(r"__launch_bounds__\([^)]*\)|__attribute__\(\(.*?\)\)\)?", "", text)
        for m in re.finditer(r"__(global|device)__[^;{}]*?\b(\w+)\s*\(([^;{}]*)\)\s*\{", text):
            depth, i = 1, m.end()
            while depth:
                depth += {"{": 1, "}": -1}.get(text[i], 0)
                i += 1
            out[m.group(2)] = (m.group(1) == "global", text[m.end():i - 1])
    return out


def _single_work_group():
    text = "".join(open(os.path.join(CSRC, f)).read() for f in FILES)
    return set(re.findall(r"hipLaunchKernelGGL\(\(?(\w+)(?:<[^>]*>)?\)?,\s*dim3\(1\)", text))


def _accesses(body):
    reads, writes = set(), set()
    for m in re.finditer(r"\bS->(\w+(?:\[[^\]]*\])?)\s*(\+=|=(?!=))?", body):
        (writes if m.group(2) else reads).add(m.group(1))
    return reads, writes


def _kernel_accesses():
    fn = _functions()

    def total(name, seen=()):
        reads, writes = _accesses(fn[name][1])
        beside = [set(), set()]           # of one work-group beside the others
        for callee in re.findall(r"\b(\w+)\s*(?:<[^;>]*>)?\(", fn[name][1]):
            if callee in fn and not fn[callee][0] and callee not in seen and callee != name:
                r, w, b = total(callee, seen + (name,))
                if callee == "pcg_check_block":
                    beside[0] |= r
                    beside[1] |= w
                else:
                    reads |= r
                    writes |= w
                    beside[0] |= b[0]
                    beside[1] |= b[1]
        return reads, writes, beside

    single = _single_work_group()
    return {n: total(n) for n, (kernel, _) in fn.items() if kernel and n not in single}


KERNELS = _kernel_accesses()


def test_the_scan_sees_the_solvers():
    for n in ("k_cg_update", "k_cg_p", "k_bicg_p", "k_bicg_s", "k_bicg_xr", "k_pcg_update", "k_pcg_update_lat",
              "k_pcg_p"):
        r, w, _ = KERNELS[n]
        assert r and w, n
    for n in ("k_box_smooth", "k_lattice_smooth", "k_mg_pre_init", "k_mg_pre_init_blk5"):
        assert "iter" in KERNELS[n][2][1], n


@pytest.mark.parametrize("name", sorted(n for n, (r, w, b) in KERNELS.items() if w or b[1]))
def test_no_kernel_reads_what_it_writes(name):
    reads, writes, beside = KERNELS[name]
    assert not reads & writes, reads & writes
    assert not (reads & beside[1] or writes & beside[0]), (reads & beside[1], writes & beside[0])
    # the convergence test's one work-group may read what its own thread updates,
    # never what it tests on entry
    assert not beside[0] & {w for w in beside[1] if w.startswith("done")}


@pytest.mark.parametrize("name", ["k_box_smooth", "k_lattice_smooth", "k_mg_pre_init", "k_mg_pre_init_blk5"])
def test_the_convergence_test_comes_before_the_vcycle_flag(name):
    """A launch that carries the convergence test must not look at the flag it
    writes: *done only through vcycle_done, and after the test's work-group."""
    body = _functions()[name][1]
    assert "*done" not in body
    assert body.index("pcg_check_block") < body.index("vcycle_done")


def test_arguments_are_taken_after_the_hierarchy_is_built():
    """mg_build may allocate anew what the solvers' arguments point to (the
    partial sums of a large lattice): a function that calls it takes the arguments
    after that."""
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, "context.hip")).read())
    # functions at file level: their bodies' brace stands in column 0
    bodies = re.findall(r"^\w[^\n;=]*\b(\w+)\(([^;{}]*)\)\s*\{\n(.*?)^\}", text, re.S | re.M)
    seen = 0
    for name, _, body in bodies:
        if "mg_build(c)" in body:
            seen += 1
            args = re.search(r"\b(?:cg|bicg)_args\(c", body)
            assert not args or body.rindex("mg_build(c)") < args.start(), name
    assert seen >= 5
