"""Runs a snippet against the library with the host-only HIP runtime of tests/cpp/host_only_hip.cpp in its place: what the
host side launches and allocates can then be tested without a GPU."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROLOGUE = """
import ctypes as C, json, os, sys
sys.modules["torch"] = None  # (it would bring a HIP runtime of its own)
import numpy as np
import fastlanes_amd as fa
_h = C.CDLL(os.environ["HOST_HIP"])
_h.host_hip_log.restype = C.c_char_p
def calls():
    '''What happened since the last call: (kind, rest of the line) each.'''
    out = [tuple(x.split(" ", 1)) for x in _h.host_hip_log().decode().splitlines()]
    _h.host_hip_clear()
    return out
def launches():
    '''(kernel, blocks, threads, LDS bytes, device) of the launches since the last call.'''
    rows = [c[1].split() for c in calls() if c[0] == "launch"]
    return [(r[0], *(int(v) for v in r[1:])) for r in rows]
"""


def build(folder) -> str:
    so = os.path.join(str(folder), "libhost_only_hip.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-shared", "-fPIC", "-o", so,
                    os.path.join(ROOT, "tests", "cpp", "host_only_hip.cpp")], check=True)
    return so


def run(so: str, snippet: str):
    """The value that the snippet assigns to `result`."""
    env = dict(os.environ, HOST_HIP=so, LD_PRELOAD=" ".join([so, os.environ.get("LD_PRELOAD", "")]).strip(), PYTHONPATH=ROOT)
    p = subprocess.run([sys.executable, "-c", PROLOGUE + snippet + "\nprint('RESULT', json.dumps(result))"], env=env, cwd=ROOT,
                       capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr[-2000:]
    return json.loads(p.stdout.split("RESULT ", 1)[1])
