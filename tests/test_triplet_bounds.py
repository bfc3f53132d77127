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


@pytest.mark.parametrize("length", [1, 1000, LONG - 1, LONG, LONG + 1])
@pytest.mark.parametrize("kind", ["plain", "read-only", "strided"])
def test_every_index_is_looked_at(length, kind):
    """The first and last index allowed, the ones beside them and the least one, at the first, a middle and the last entry."""
    n = 70_000
    good = np.random.default_rng(length).integers(0, n, size=length).astype(np.int32)
    data = np.ones(length, dtype=np.float32)
    for place in {0, length // 2, length - 1}:
        for value in (0, n - 1, n, -1, -2**31):
            index = good.copy()
            index[place] = value
            if kind == "read-only":
                index.flags.writeable = False
            elif kind == "strided":
                index = np.repeat(index, 2)[::2]
            inside = 0 <= value < n
            assert fmm._inside(index, n) == inside
            for row, col in ((index, good), (good, index)):
                assert fmm._are_plain_triplets(row, col, data, (n, n)) == inside
                if inside:
                    assert MTX.from_coo(row, col, (n, n), data=data).num_edges() == length
                else:
                    with pytest.raises(ValueError):
                        MTX.from_coo(row, col, (n, n), data=data)


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
