"""Host cost of launch planning: the rules ask for the compute units of the current device many times
per call, the runtime is asked once (each question costs 30-50 ns of a 4-8 us call)."""
import os
import subprocess
import sys

from rl_triton import _native

COUNTING = r"""
static int calls;
int hipGetDevice(int *device) { ++calls; *device = 0; return 0; }
int hipDeviceGetAttribute(int *value, int attribute, int device) { (void)attribute; (void)device; *value = 256; return 0; }
int device_questions(void) { return calls; }
"""

CHILD = r"""
import ctypes, sys
counting = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # ahead of the runtime's own
lib = ctypes.CDLL(sys.argv[2])
f = lib.rlk_gae_normalized_partials_bytes
f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_int64] * 2
for shape in [(64, 64), (4096, 128), (8, 16313), (3, 40000), (16, 131072), (300, 7000), (4096, 2561)]:
    before = counting.device_questions()
    assert f(*shape) > 0
    print(shape, counting.device_questions() - before)
"""


def test_the_device_is_asked_for_once_per_planning_step(tmp_path):
    src, so = tmp_path / "counting.c", tmp_path / "counting.so"
    src.write_text(COUNTING)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so)], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD, str(so), os.path.abspath(_native.library_path())],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    counts = [int(line.rsplit(" ", 1)[1]) for line in r.stdout.splitlines()]
    assert len(counts) == 7 and all(n == 1 for n in counts), r.stdout
