"""The bounds of triplet arrays (MTX.from_coo): one thread or torch's, and the processes that must not use those."""
import multiprocessing
import os
import subprocess
import sys

import numpy as np
import pytest

from liteform_ae_amd import format_matrix_market as fmm
from liteform_ae_amd.format_matrix_market import MTX

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LONG = fmm._BY_THREADS


def _in_child(answers, index):
    answers.put(MTX.from_coo(index, index, (LONG, LONG)).num_edges())


def test_a_forked_process_does_not_wait_for_its_parents_threads():
    torch = pytest.importorskip("torch")
    if torch.cuda.is_initialized():
        pytest.skip("a process that uses the GPU is not forked")
    index = np.arange(LONG, dtype=np.int32)
    torch.aminmax(torch.arange(4 * LONG))                      # the parent's threads are there
    context = multiprocessing.get_context("fork")
    answers = context.Queue()
    child = context.Process(target=_in_child, args=(answers, index))
    child.start()
    child.join(60)
    stuck = child.is_alive()
    if stuck:
        child.kill()
        child.join()
    assert not stuck and answers.get(timeout=10) == LONG


def test_a_process_without_torch_stays_without():
    program = ("import sys, numpy as np\n"
               "from liteform_ae_amd.format_matrix_market import MTX\n"
               f"index = np.arange({LONG}, dtype=np.int32)\n"
               f"assert MTX.from_coo(index, index, ({LONG}, {LONG})).num_edges() == {LONG}\n"
               "assert 'torch' not in sys.modules")
    subprocess.run([sys.executable, "-c", program], check=True, timeout=120, cwd=ROOT)
