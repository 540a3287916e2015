"""Runs a script against the engine on tests/fake_hip_runtime.c, in a process
of its own (the fake runtime has to be loaded before the engine)."""
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for f in (fake.fake_largest, fake.fake_live):
    f.restype = ctypes.c_size_t
fake.fake_set_limit.argtypes = fake.fake_set_capacity.argtypes = [ctypes.c_size_t]
sys.path.insert(0, sys.argv[2])
import numpy as np
import steps_amd as steps
fake.fake_launches.restype = ctypes.c_long
def launches(part, blocks=0):
    return fake.fake_launches(part.encode(), blocks)
NO_LIMIT = (1 << 64) - 1
def cloud(N, L=None):
    rng = np.random.default_rng(N)
    x = rng.normal(size=(N, 3)) * 30.0 if L is None else rng.uniform(0.0, L, (N, 3))
    return x, np.ones(N), np.full(N, 0.01)
def code(call):
    try:
        call()
        return 0
    except steps.StepsError as e:
        return e.code
"""


def run(tmp_path, script, timeout=120):
    """The script's output lines."""
    so = tmp_path / "libfakehip.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(so), str(HERE / "fake_hip_runtime.c")], check=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE + script, str(so), str(HERE.parent)], capture_output=True,
                       text=True, timeout=timeout)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout.splitlines()
