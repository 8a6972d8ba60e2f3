"""Constant memory (address space 4) promises the compiler that a value does
not change while the kernel runs, so that it may load it again at any time.
Every kernel that reads fields of a group's control block that way leaves
those fields alone."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "steadyscan_amd", "csrc",
                   "ss_kernels.hip")


def functions(text):
    """(name, body) of every function definition."""
    for m in re.finditer(r"^[A-Za-z_][^;{}=]*?\b(\w+)\([^;{}()]*\)\s*\{\n", text, re.M):
        yield m.group(1), text[m.end():text.index("\n}\n", m.end())]


def const_fields(body):
    """Fields of the control block read through constant memory."""
    direct = set(re.findall(r"as_const\(B\.ctl\)\[\w+\]\.(\w+)", body))
    for alias in re.findall(r"const SS_CONST GroupCtl &(\w+) = as_const\(B\.ctl\)", body):
        direct |= set(re.findall(r"\b%s\.(\w+)" % alias, body))
    return direct


def written_fields(body, called):
    """Fields assigned here or in the functions called with the control block."""
    out = set(re.findall(r"\b(?:ctl|out|c)\.(\w+)\s*(?:[-+|&]?=)(?!=)", body))
    out |= set(re.findall(r"atomic\w+\(&(?:ctl|out)\.(\w+)", body))
    for name in called:
        if re.search(r"\b%s\(" % name, body):
            out |= called[name]
    return out


def test_no_kernel_writes_what_it_reads_as_constant():
    text = re.sub(r"//[^\n]*", "", open(SRC).read())
    bodies = dict(functions(text))
    helpers = {n: written_fields(bodies[n], {}) for n in ("stage_time", "final_finish", "ls_decide_frame")}
    assert {"phase"} <= helpers["final_finish"] and {"tStage"} <= helpers["stage_time"]
    kernels = [n for n in bodies if n.startswith("k_")]
    assert {"k_assemble", "k_solve", "k_ls_round", "k_ls_decide", "k_ls_finish", "k_corr_finish"} <= set(kernels)
    for name in kernels:
        both = const_fields(bodies[name]) & written_fields(bodies[name], helpers)
        assert not both, (name, both)
    assert const_fields(bodies["k_ls_decide"]) >= {"phase", "shift", "roundsThisLS"}
