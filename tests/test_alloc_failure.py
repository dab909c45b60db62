"""An allocation that fails is reported and leaves the handle usable.  Runs the
library's host code on the CPU over a HIP runtime (fake_hip.cpp) whose launches
do nothing and whose next allocation of a given size can be made to fail; a
launch that would be given memory that is not there is seen in its arguments."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = "/opt/rocm"

START = r"""
import ctypes, sys
sys.path.insert(0, sys.argv[2])
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # before the library's own runtime
fake.fake_fail.argtypes = [ctypes.c_size_t]
import torch_amd as ta
from torch_amd import surrogate as sg

cool = ta.Cooling(ta.thermo_params(), stream=0)
mlp = sg.MLP(max_batch=32, stream=0)
sg.set_surrogate(cool, mlp, sg.make_cfg([0] * 8, [1] * 8, [-1e30] * 6, [1e30] * 6))
n = 100
buf = (ctypes.c_double * (14 * n))()
at = ctypes.addressof(buf)
grid = ta.Grid(ta.make_params((8, 8, 8), bc="free"), stream=0)

def substep():
    return ta.lib().torchgpu_thermo_grid_substep(grid._h, cool._h, None, None, None, -1, ctypes.c_double(1.0), 0)

def surrogate():
    fake.fake_watch(b"surrogate_prepass", 11)   # fb_list
    rc = ta.lib().torchgpu_thermo_cells_surrogate(cool._h, n, at, at + 9 * 8 * n, None, None)
    assert fake.fake_launches() == (1 if rc == 0 else 0)
    return rc

"""

QUEUE = START + r"""
assert surrogate() == 0 and fake.fake_seen_live()
fake.fake_fail(8 * 512)            # the fallback queue of the grid's 512 cells
substep()
assert surrogate() == 0 and fake.fake_seen_live(), "the prepass writes through a freed queue"
assert substep() == 0
assert surrogate() == 0 and fake.fake_seen_live()
print("done")
"""

# The FP64 grid step and loop ran in less memory before they had a queue and
# kept rates: without those they gather the inputs and form the rates again.
LIMIT = START + r"""
fake.fake_fail(8 * 512)
fake.fake_watch(b"thermo_gather", 1)
assert substep() == 0 and fake.fake_launches() == 1
fake.fake_watch(b"thermo_gather", 1)
assert substep() == 0 and fake.fake_launches() == 0   # memory again: the direct step
fake.fake_fail(16 * 512)
fake.fake_watch(b"thermo_timestep", 8)   # the kept rates
cool.run_split(grid, 2)
assert fake.fake_launches() == 2 and fake.fake_seen_live() == 0
fake.fake_watch(b"surrogate_prepass", 17)
cool.run_split(grid, 2)
assert fake.fake_launches() == 3   # one step opens with the cooling, the other closes with two halves
print("done")
"""


@pytest.mark.parametrize("script", [QUEUE, LIMIT], ids=["queue", "limit"])
def test_failed_allocation(tmp_path, script):
    so = str(tmp_path / "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", so], check=True)
    r = subprocess.run([sys.executable, "-c", script, so, ROOT], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout + r.stderr
