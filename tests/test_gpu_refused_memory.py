"""Calls on a device that has less memory than they ask for.  Each case runs in a
process of its own in front of whose library allocation functions stand that
answer out-of-memory for a range of sizes (refuse_alloc/refuse.c).

Each test prints its case before the GPU work starts.
"""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = tmp_path_factory.mktemp("refuse") / "refuse.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", os.path.join(HERE, "refuse_alloc", "refuse.c"), "-o", str(so),
                    "-ldl"], check=True)
    return so


@pytest.mark.parametrize("case", ["one_pass", "one_pass_plain", "one_pass_graph", "host_arrays_pinned",
                                  "host_arrays_pinned_later", "host_arrays_device"])
def test_refused_memory(shim, case):
    print(f"case: {case}", flush=True)
    env = dict(os.environ, PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, os.path.join(HERE, "refuse_alloc", "child.py"), str(shim), case], cwd=ROOT,
                       env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("same\n"), r.stdout + r.stderr
