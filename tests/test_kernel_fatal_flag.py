"""The kernels' early exit on a fatal flag, by their source: a workgroup whose waves meet at a barrier
must leave as one where its own launch may raise such a flag, because other workgroups raise it while
this one starts, and a wave that stayed alone would use LDS that the others were to set.  Such
kernels take one thread's reading for all (workgroup_fatal); one wave at a time, or flags that no
workgroup of the launch raises, may be read per wave (batch_fatal)."""
import os
import re

import openmmcustomgbintegralforce_amd as pkg

CSRC = os.path.join(os.path.dirname(pkg.__file__), "csrc")


def _fatal_names():
    text = open(os.path.join(CSRC, "gbi_internal.h")).read()
    return set(re.findall(r"FLAG_\w+", re.search(r"kFatalFlags\s*=(.*?);", text, re.S).group(1)))


def _kernels():
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, "gbi_kernels.hip")).read())
    for m in re.finditer(r"__global__\s+void\s+(?:__launch_bounds__\((?P<b>(?:[^()]|\([^()]*\))*)\)\s*)?(?P<n>\w+)\(", text):
        body = text[m.end():text.index("\n}\n", m.end())]
        yield m.group("n"), (m.group("b") or "").split(",")[0].strip(), body


def test_workgroups_leave_as_one():
    fatal, seen, wrong = _fatal_names(), [], []
    assert "FLAG_POINT_OVERFLOW" in fatal and "FLAG_NONFINITE_RESULT" not in fatal
    for name, threads, body in _kernels():
        raises = any(f in body for f in fatal)
        if threads == "64" or "__syncthreads()" not in body or not raises:
            continue
        seen.append(name)
        if "batch_fatal(" in body.replace("workgroup_fatal(", "") or "workgroup_fatal(" not in body:
            wrong.append(name)
    assert set(seen) == {"k_gbsw_points", "k_point_bin", "k_point_split", "k_worklist"}
    assert not wrong, wrong
