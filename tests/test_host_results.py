"""Page-locked buffers of a design's logits (stage._PinnedResults), with a library that only keeps account of them."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from glinthawk_amd import _lib, stage

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class Account:
    def __init__(self):
        self.memory, self.freed = [], []
        self.gh_host_free = self.freed.append

    def gh_host_malloc(self, out, n_bytes):
        self.memory.append((C.c_char * n_bytes)())
        out._obj.value = C.addressof(self.memory[-1])
        return 0


@pytest.fixture
def account(monkeypatch):
    a = Account()
    monkeypatch.setattr(_lib, "lib", lambda: a)
    return a


def test_closing_releases_what_is_not_in_use(account):
    """The buffers in use stay with their arrays, views included, and each goes with its own."""
    pool = stage._PinnedResults(4 * 6, 2)
    places = [C.addressof(m) for m in account.memory]
    a = pool.take(2, 3)
    a[:] = 7
    view = a[1:, ::2]
    mine = a.ctypes.data
    assert mine in places and account.freed == []
    pool.close()
    assert account.freed == [p for p in places if p != mine] and pool.take(2, 3) is None
    del a
    assert len(account.freed) == 1 and (view == 7).all()
    del view
    assert sorted(account.freed) == sorted(places)
    del pool
    assert len(account.freed) == 2


def test_a_dropped_pool_releases_everything_once(account):
    pool = stage._PinnedResults(64, 2)
    a, b = pool.take(4, 4), pool.take(1, 1)
    assert pool.take(1, 1) is None and pool.take(5, 4) is None
    del b
    c = pool.take(2, 2)
    assert isinstance(c, np.ndarray) and account.freed == []
    del pool
    assert account.freed == []
    del a, c
    assert len(account.freed) == len(set(account.freed)) == 2


def test_the_interpreter_ends_with_arrays_in_use():
    """The program's own names go last where something holds its module: those of the package are gone then."""
    code = """
import sys
from glinthawk_amd import _lib, stage
from test_host_results import Account
account = Account()
_lib.lib = lambda: account
pool = stage._PinnedResults(64, 3)
array = pool.take(4, 4)
sys.keep = sys.modules["__main__"]
"""
    done = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env={**os.environ, "PYTHONPATH": os.pathsep.join([ROOT, os.path.join(ROOT, "tests")])}, capture_output=True, text=True,
                          timeout=100)
    assert done.returncode == 0 and done.stderr == "", done.stderr
