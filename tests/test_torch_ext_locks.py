"""The chain workspaces that the PyTorch extension remembers are Python's tensors:
no thread may hold the cache's mutex while it waits for the interpreter lock."""

from __future__ import annotations

import os
import subprocess
import sys

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "nanochat-filter_amd")

_RACE = """
import threading, time, torch
from nanochat_amd import _native as N
ext = N.torch_ext()
stop = threading.Event()
def grow():
    # every buffer but the newest is owned by the cache alone: replacing one
    # frees its Python object
    while not stop.is_set():
        _, drops = ext._find_chain_workspace(0, 1, 1 << 40)
        ext._keep_chain_workspace(0, 1, torch.zeros(256, dtype=torch.uint8), drops)
t = threading.Thread(target=grow, daemon=True)
t.start()
for _ in range(2000):
    time.sleep(0.0005)  # several buffers are replaced between two drops
    ext.drop_chain_workspaces()
stop.set()
t.join()
print("done")
"""


def test_dropping_while_another_thread_remembers():
    env = dict(os.environ, PYTHONPATH=PKG)
    p = subprocess.run([sys.executable, "-c", _RACE], env=env, capture_output=True, text=True,
                       timeout=100)
    assert p.returncode == 0 and p.stdout.strip() == "done", p.stderr


def test_a_dropped_workspace_is_not_remembered_again():
    torch = pytest.importorskip("torch")
    sys.path.insert(0, PKG)
    from nanochat_amd import _native as N

    ext = N.torch_ext()
    key = (7, 0x1230)
    buf = torch.zeros(512, dtype=torch.uint8)
    none, drops = ext._find_chain_workspace(*key, 512)
    assert none is None
    ext.drop_chain_workspaces()  # another thread's error, while buf was being made
    ext._keep_chain_workspace(*key, buf, drops)
    assert ext._find_chain_workspace(*key, 512)[0] is None
    ext._keep_chain_workspace(*key, buf, ext._find_chain_workspace(*key, 512)[1])
    kept = ext._find_chain_workspace(*key, 512)[0]
    assert kept is not None and kept.data_ptr() == buf.data_ptr()
    assert ext._find_chain_workspace(*key, 513)[0] is None
    ext.drop_chain_workspaces()
    assert ext._find_chain_workspace(*key, 1)[0] is None
