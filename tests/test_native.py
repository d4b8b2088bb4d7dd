"""The C++ template API through small programs (tests/native/*.hip, built by
kites_amd.build): value types, functor forms and call counts that the C ABI's
fixed functor sets do not reach.  Each program prints the case before it runs
and checks it against a host reference of its own."""
import os
import subprocess

import pytest

from conftest import ROOT, case

BUILD = os.path.join(ROOT, "tests", "native", "_build")


def _run(name, *args, timeout=110):
    exe = os.path.join(BUILD, name)
    assert os.path.exists(exe), "native tests not built (python -m kites_amd.build)"
    case(" ".join((name,) + args))
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=timeout)
    print(r.stdout[-6000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0 and "all checks passed" in r.stdout and "FAILED" not in r.stdout
    return r.stdout


def test_headers_on_the_host():
    _run("host_forms")


@pytest.mark.gpu
def test_ordered_value_types():
    out = _run("ordered_types")
    assert out.count("ok:") == 20


@pytest.mark.gpu
def test_functor_forms():
    out = _run("functor_forms")
    assert out.count("ok:") == 8 * 2 * 21


@pytest.mark.gpu
def test_edge_pointer():
    out = _run("edge_pointer")
    assert out.count("ok:") == 10


@pytest.mark.gpu
def test_volatile_sets():
    out = _run("volatile_sets")
    assert out.count("ok:") == 2 * (2 * 17 + 2 * 13 + 2 * 2 + 2)
