"""The share of rows that leave the first path of a top-k call, as bench.py reports it: the first path
follows from the batch's size, never from which path the rows were seen to take."""
import os
import re
import sys
from types import SimpleNamespace

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402


def rate(paths, rows, n_vocab):
    hs = SimpleNamespace(sample=lambda *a: None, topk_paths=lambda n: np.array(paths[:n]))
    return bench.topk_path_counts(hs, [SimpleNamespace(n_vocab=n_vocab)], None, None, None,
                                  rows)["fallback_rate"]


@pytest.mark.parametrize("rows,n_vocab,paths,want", [
    (64, 128256, [0] * 64, 0.0),                     # all served by the candidates
    (64, 128256, [1] * 64, 1.0),                     # all of them fell back to the thread maxima
    (64, 128256, [0] * 48 + [1] * 12 + [2] * 4, 0.25),
    (256, 262144, [1] * 256, 0.0),                   # thread maxima first
    (128, 131072, [1] * 128, 1.0), (256, 131072, [1] * 256, 0.0), (127, 131073, [1] * 127, 1.0),
    (128, 131073, [1] * 128, 0.0),
    (256, 262144, [1] * 192 + [2] * 64, 0.25),
])
def test_fallback_rate(rows, n_vocab, paths, want):
    assert rate(paths, rows, n_vocab) == want


def test_the_limit_is_the_librarys():
    text = open(os.path.join(ROOT, "geistlib_amd", "csrc", "sampler_kernels.h")).read()
    chunks, long_rows, others = re.search(r"1 << \(n_chunks > (\d+) \? (\d+) : (\d+)\)", text).groups()
    assert bench.TOPK_MAXIMA_ROW == int(chunks) * 8192
    assert bench.TOPK_MAXIMA_LOGITS == (1 << int(long_rows), 1 << int(others))
