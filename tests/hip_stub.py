"""Child processes that load libcmf_hip.so over the stand-in of the HIP runtime
(hip_stub.c), so that what the host side does can be tested without a GPU."""
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

HEAD = """
import ctypes, json, sys
stub = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = [{root!r}, {pkg!r}, {here!r}]
stub.stub_fail(0, 0, 0, 0)
def result(x):
    print("RESULT " + json.dumps(x), flush=True)
"""


def run(tmp_path, code, source="hip_stub.c", timeout=300):
    """The value that `code` hands to result()."""
    lib = str(tmp_path / "stub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", os.path.join(HERE, source), "-o", lib, "-ldl"], check=True)
    head = HEAD.format(lib=lib, root=ROOT, pkg=os.path.join(ROOT, "cama-flood_v4_amd"), here=HERE)
    p = subprocess.run([sys.executable, "-c", head + code], capture_output=True, text=True, timeout=timeout)
    assert p.returncode == 0, f"exit {p.returncode}\n{p.stdout[-2000:]}\n{p.stderr[-4000:]}"
    lines = [x[7:] for x in p.stdout.splitlines() if x.startswith("RESULT ")]
    assert len(lines) == 1, p.stdout[-2000:]
    return json.loads(lines[0])
