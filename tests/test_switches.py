"""Switches are read from the environment when the kernels are first needed,
not when the package is imported."""
import subprocess
import sys


def test_a_program_may_set_them_after_its_imports():
    # a process of its own, which has not needed the kernels yet
    subprocess.run([sys.executable, "-c", """
import os
from ollamamq_amd import engine, models
from ollamamq_amd.ops import interface
os.environ["OLLAMAMQ_NO_WSTREAM"] = "1"
os.environ["OLLAMAMQ_WS_KS"] = "3"
assert interface.library_products()
assert interface.asked_parts(4096) == 3
from ollamamq_amd.ops import hip
assert interface.hip is hip
"""], check=True)
