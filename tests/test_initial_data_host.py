"""What the generator of initial states leaves behind on the host: no threads that go on waiting
actively. A program copies or converts the state next, on the same cores."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import time
from ctf_amd import native
native.init_turbulence((48, 48, 48), v_rms=0.3, dB_rms=0.3, seed=1)
before = time.process_time()
time.sleep(0.15)
print(time.process_time() - before)
"""


def test_no_thread_spins_after_the_generator():
    """CPU time of the process over 0.15 s of sleep: next to none (an OpenMP team of two that
    waits actively takes 0.15 s)."""
    env = dict(os.environ, OMP_NUM_THREADS="4", PYTHONPATH=ROOT)
    out = subprocess.run([sys.executable, "-c", PROGRAM], cwd=ROOT, env=env, capture_output=True, text=True, check=True)
    assert float(out.stdout) < 0.05
