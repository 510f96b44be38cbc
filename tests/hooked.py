"""Runs a piece of Python in a child process with the HIP entry points of
hip_hooks.c in front of the runtime's."""
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
HEAD = """
import ctypes, sys
sys.path[:0] = [%r, %r, %r]
hooks = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
hooks.hook_count.restype = ctypes.c_long
PINNED, MALLOC, MEMCPY, MEMSET = range(4)
"""


def run(code, timeout=100, **env):
    """What the child prints (its last line)."""
    root = os.path.dirname(HERE)
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "hip_hooks.so")
        subprocess.run(["gcc", "-O1", "-w", "-shared", "-fPIC", "-o", so,
                        os.path.join(HERE, "hip_hooks.c"), "-ldl"],
                       check=True)
        r = subprocess.run(
            [sys.executable, "-u", "-c",
             HEAD % (root, HERE, os.path.join(root, "oracle"), so) + code],
            env=dict(os.environ, **env), stdout=subprocess.PIPE, text=True,
            timeout=timeout)
    assert r.returncode == 0, r.stdout[-2000:]
    return r.stdout.strip().splitlines()[-1]
