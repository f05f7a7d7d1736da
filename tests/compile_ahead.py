"""Compiles kernels into the code-object cache side by side, for tests that take many: hipRTC compiles one at a time in a process (a
lock of its own), so this takes several, which emit and compile and touch no GPU."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WORKER = """
import json, sys
from kernelcodegen_amd import runtime as R
for family, params in json.load(sys.stdin):
    R.compile_to_code(R.prelude() + R.emit_kernel(family, "kernel0", **R.launch_params(family, params))[0])
"""


def compile_ahead(kernels, workers=8):
    """`kernels`: (family, parameters) as runtime.get_kernel takes them."""
    running = [subprocess.Popen([sys.executable, "-c", WORKER], cwd=ROOT, stdin=subprocess.PIPE, text=True) for _ in range(workers)]
    for i, process in enumerate(running):
        process.stdin.write(json.dumps(kernels[i::workers]))
        process.stdin.close()
    assert not any([process.wait() for process in running])
