"""A kernel that leaves early because the job overflowed looks only at bits that
earlier launches raised. A bit that its own workgroups raise can go up between two
waves' loads of it: some waves of a workgroup would leave, and the others go on
with LDS that those never wrote."""
import os
import re

import pytest

from rusterizer_amd import build


def _kernels():
    text = open(os.path.join(build.CSRC, "rz_kernels.hip")).read()
    text = re.sub(r"//.*", "", text)
    out = {}
    for m in re.finditer(r"__global__[^;{]*?void\s+(?:__attribute__\(\(.*?\)\)\s*)?(k_\w+)\(", text, re.S):
        i = text.index("{", m.end())
        depth, j = 1, i + 1
        while depth:
            depth += {"{": 1, "}": -1}.get(text[j], 0)
            j += 1
        out[m.group(1)] = text[i:j]
    return out


KERNELS = _kernels()


def _bits(expr):
    return set(re.findall(r"OVF_\w+", expr))


@pytest.mark.parametrize("name", ["k_setup", "k_bin", "k_fine_bin", "k_tile_bin"])
def test_kernel_does_not_leave_on_a_bit_it_raises(name):
    body = KERNELS[name]
    raised = set().union(*map(_bits, re.findall(r"atomicOr\(&b\.cnt->overflow,([^;]*)\)", body)))
    assert raised, name
    assert "b.cnt->overflow" not in re.sub(r"atomicOr\(&b\.cnt->overflow", "", body), name
    exits = re.findall(r"if \(job_stopped\(b,([^;]*)\)\) return;", body)
    assert len(exits) == 1 and raised <= _bits(exits[0]), (name, raised, exits)
