"""The native module's workspace and Python threads (on the CPU)."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# A dispatch mode runs Python inside the allocations of the thread that
# switched it on, and so lets other threads run in the middle of a call.
SCRIPT = """
import threading, time, torch
from torch.utils._python_dispatch import TorchDispatchMode
from bitsparse_amd import _lib

ws = _lib.native().Workspace(torch.device("cpu"))
ws.ensure(1 << 10)
ws.buf[:8] = torch.arange(8, dtype=torch.uint8)
seen = []


class Slow(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        seen.append(str(func))
        time.sleep(0.2)
        return func(*args, **(kwargs or {}))


def grow():
    with Slow():
        ws.ensure(1 << 20)
        ws.epoch = (1 << 30) - 1
        ws.next_epoch(2)                 # (cleared: the counter wraps)


t = threading.Thread(target=grow)
t.start()
time.sleep(0.1)
ws.ensure(1 << 18)                       # a second thread meets the first one in its allocation
ws.next_epoch()
t.join()
assert ws.nbytes >= 1 << 20
assert not seen, seen                    # the workspace is no business of the thread's modes
print("done")
"""


def test_workspace_calls_meet_without_a_hang():
    r = subprocess.run([sys.executable, "-c", SCRIPT], cwd=ROOT, capture_output=True, text=True, timeout=90)
    assert r.returncode == 0 and r.stdout.strip() == "done", r.stdout + r.stderr
