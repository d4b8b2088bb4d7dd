"""Orderings that only the generated gfx950 code shows (compiled here, no
GPU): a barrier of a workgroup waits for no load in flight."""
import os
import re
import subprocess

import pytest

from conftest import ROOT
from kites_amd import build


@pytest.fixture(scope="module")
def persist_code(tmp_path_factory):
    try:
        cc = build.hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    out = tmp_path_factory.mktemp("isa") / "persist_loop.s"
    subprocess.run([cc, *[f for f in build.HIP_FLAGS if f != "-fPIC"], "-I", build.CSRC, "-S",
                    "--cuda-device-only", os.path.join(ROOT, "tests", "isa", "persist_loop.hip"),
                    "-o", str(out)], check=True, capture_output=True, timeout=300)
    return out.read_text()


def test_loop_reads_before_it_relaxes(persist_code):
    """The one-workgroup loop's first barrier separates the reads of the values
    an iteration starts from and the atomics that lower them: every load has
    returned (vmcnt 0) before each such barrier."""
    found = 0
    for body in re.findall(r"^_ZN5kites6detail14persist_kernel\S*:.*?^\s*s_endpgm.*?^\.Lfunc_end",
                           persist_code, re.M | re.S):
        code = [l.strip() for l in body.splitlines()]
        barriers = [i for i, l in enumerate(code) if l.startswith("s_barrier")]
        for b, nxt in zip(barriers, barriers[1:] + [len(code)]):
            if not any(l.startswith("global_atomic_umin") for l in code[b:nxt]):
                continue
            found += 1
            prev = max((i for i in barriers if i < b), default=0)
            last = [l for l in code[prev:b] if l.startswith("global_load") or "vmcnt(0)" in l][-1:]
            assert last and "vmcnt(0)" in last[0], code[max(0, b - 8):b + 1]
    assert found == 8      # plain and near-far, one to four edges per thread
