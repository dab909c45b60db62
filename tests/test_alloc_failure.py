"""An allocation that fails is reported and leaves the handle usable.  Runs the
library's host code on the CPU over a HIP runtime (fake_hip.cpp) whose launches
do nothing and whose next allocation of a given size can be made to fail; a
launch that would be given memory that is not there is seen in its arguments."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = "/opt/rocm"

SCRIPT = r"""
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

def surrogate():
    fake.fake_watch(b"surrogate_prepass", 11)   # fb_list
    rc = ta.lib().torchgpu_thermo_cells_surrogate(cool._h, n, at, at + 9 * 8 * n, None, None)
    assert fake.fake_launches() == (1 if rc == 0 else 0)
    return rc

assert surrogate() == 0 and fake.fake_seen_live()
grid = ta.Grid(ta.make_params((8, 8, 8), bc="free"), stream=0)
fake.fake_fail(8 * 512)            # the fallback queue of the grid's 512 cells
assert ta.lib().torchgpu_thermo_grid_substep(grid._h, cool._h, None, None, None, -1, ctypes.c_double(1.0), 0) == 2
assert surrogate() == 0 and fake.fake_seen_live(), "the prepass writes through a freed queue"
assert ta.lib().torchgpu_thermo_grid_substep(grid._h, cool._h, None, None, None, -1, ctypes.c_double(1.0), 0) == 0
assert surrogate() == 0 and fake.fake_seen_live()
print("done")
"""


def test_fallback_queue_after_a_failed_allocation(tmp_path):
    so = str(tmp_path / "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", so], check=True)
    r = subprocess.run([sys.executable, "-c", SCRIPT, so, ROOT], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout + r.stderr
