"""The host side of calls issued natively, each case in a process with a stand-in for the library (recording_cases.py)."""
import ast
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CASES = [n.name for n in ast.parse(open(os.path.join(HERE, "recording_cases.py")).read()).body
         if isinstance(n, ast.FunctionDef) and not n.args.args and not n.args.vararg]


@pytest.mark.parametrize("case", CASES)
def test_recording(case):
    path = os.pathsep.join([os.path.dirname(HERE), HERE])
    done = subprocess.run([sys.executable, os.path.join(HERE, "recording_cases.py"), case], env={**os.environ, "PYTHONPATH": path},
                          capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout + done.stderr
