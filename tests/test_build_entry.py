"""build() takes the test suite's programs from whichever of its modules are
there: an older test tree, or none, still builds the product."""
import os
import shutil
import subprocess
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
COLLECT = ("import sys; sys.path.insert(0, %r); import __graft_entry__ as g; "
           "print(' '.join(name for name, _, _ in g.build_tests_programs(%r)))")


@pytest.mark.parametrize("modules", [(), ("randprog",), ("tileprog",), ("randprog", "tileprog"), None])
def test_programs_of_the_modules_that_are_there(tmp_path, modules):
    tests = tmp_path / "tests"  # None: no test tree at all
    if modules is not None:
        tests.mkdir()
    for m in modules or ():
        shutil.copy(os.path.join(REPO, "tests", m + ".py"), tests)
    r = subprocess.run([sys.executable, "-c", COLLECT % (REPO, str(tests))], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    names = r.stdout.split()
    assert any(n.startswith("rand_") for n in names) == ("randprog" in (modules or ()))
    assert ("ew_tr3_ragged" in names) == ("tileprog" in (modules or ()))
