"""The bounds of triplet arrays (MTX.from_coo): one thread or torch's, and the processes that must not use those."""
import multiprocessing

import numpy as np
import pytest

from liteform_ae_amd import format_matrix_market as fmm
from liteform_ae_amd.format_matrix_market import MTX

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
