"""The stop flags of the solvers whose kernels decide on the device.

Blocks of one launch start at any time, and the waves of a block read for
themselves: where one thread of a launch stores a flag that others load, some
waves of a block may return and the others go on into a block-wide barrier.
So no kernel of more than one block may read a stop flag that it (or a device
function that it calls) writes.  Checked on the source: the flags are the
fields stop, stop_seen of the device states (FoldHost, written for the host, is
not read by kernels)."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "modflow6_amd", "csrc")
FIELD = r"\b(?!hf\b)(\w+)->(stop\w*)\b"


def functions(text):
    """name -> (is a kernel, body) of every device function of a source."""
    out = {}
    for m in re.finditer(r"__(global|device)__\b([^;{}]*?)\b(\w+)\s*\(", text):
        if m.group(3).startswith("__launch_bounds"):
            continue
        at = text.index("{", m.end())
        depth, end = 1, at + 1
        while depth:
            depth += {"{": 1, "}": -1}.get(text[end], 0)
            end += 1
        out[m.group(3)] = (m.group(1) == "global", text[at:end])
    return out


def kernels(name):
    """(kernel, flags read, flags written) of a source; a template over bool Q
    counts once per value, one-block kernels are left out."""
    with open(os.path.join(CSRC, name)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    text = re.sub(r"__launch_bounds__\s*\([^()]*(\([^()]*\)[^()]*)*\)", "", text)
    funcs = functions(text)
    one_block = set(re.findall(r"\b(\w+)(?:<[^<>;]*>)?<<<1,", text))
    for k, (is_kernel, body) in funcs.items():
        if not is_kernel or k in one_block:
            continue
        for q in ("false", "true") if re.search(r"\bQ \?|!Q\b", body) else ("",):
            b = body
            if q:
                b = re.sub(r"\bQ \? ([^:;]+) : ([^;,)]+)", r"\1" if q == "true" else r"\2", b)
            if q == "true":     # the blocks that run the test belong to Q false
                b = re.sub(r"if \(!Q &&[^{}]*\{(?:[^{}]|\{[^{}]*\})*\}", "", b)
            seen, todo = set(), [b]
            reads, writes = set(), set()
            while todo:
                t = todo.pop()
                writes |= {w[:2] for w in re.findall(FIELD + r"\s*=(?!=)", t)}
                reads |= set(re.findall(FIELD + r"(?!\s*=[^=])", t))
                for callee in re.findall(r"\b(\w+)(?:<[^<>;]*>)?\s*\(", t):
                    if callee in funcs and callee not in seen and not funcs[callee][0]:
                        seen.add(callee)
                        todo.append(funcs[callee][1])
            yield k + (f"<Q {q}>" if q else ""), reads, writes


@pytest.mark.parametrize("name", ["mf6hip_cgfold.hip", "mf6hip_bcgsfold.hip", "mf6hip_fcg.hip"])
def test_no_kernel_reads_the_stop_flag_it_writes(name):
    some_read, some_written = set(), set()
    for k, reads, writes in kernels(name):
        assert not reads & writes, (k, reads & writes)
        some_read |= reads
        some_written |= writes
    # the flags were found: a solver that stops by itself has both
    assert some_read and some_written
