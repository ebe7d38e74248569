"""An FP32 upload that runs out of host memory returns an error: no exception
leaves the C entry point and no helper thread ends the process, wherever the
allocation fails."""

import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# argv: view, MiB of address space left for the upload (which needs several hundred)
PROGRAM = """
import ctypes, resource, sys
from trajsparsenufft_amd import pack, synth
from trajsparsenufft_amd._lib import lib
from trajsparsenufft_amd.pack import KbMatrix
kb = KbMatrix.build(synth.radial(800, 512), (256, 256), (512, 512))
out, entry = ctypes.c_void_p(), lib().tsn_direction_upload_csr
in_use = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (in_use + int(sys.argv[2]) * 2**20, resource.RLIM_INFINITY))
rc = entry(kb.handle, int(sys.argv[1]), ctypes.byref(out))
resource.setrlimit(resource.RLIMIT_AS, (resource.RLIM_INFINITY, resource.RLIM_INFINITY))
assert rc != 0 and not out.value, (rc, out.value)
print(lib().tsn_last_error().decode())
"""


@pytest.mark.parametrize("view,room", [(0, 1), (0, 60), (0, 120), (1, 1), (1, 60), (1, 120), (1, 210)])
def test_upload_without_memory_is_an_error(view, room):
    # (freed memory goes back at once, so that the limit holds from the first array on)
    env = dict(os.environ, MALLOC_MMAP_THRESHOLD_="131072", MALLOC_ARENA_MAX="1")
    run = subprocess.run([sys.executable, "-c", PROGRAM, str(view), str(room)], cwd=ROOT, capture_output=True,
                         text=True, timeout=120, env=env)
    assert run.returncode == 0, (run.returncode, run.stderr[-500:])
    assert "out of host memory" in run.stdout
