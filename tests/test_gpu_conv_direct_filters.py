"""First layers whose filters end in odd places: fewer elements than a 16-byte piece in all, runs of one piece and of several, an odd
and an even number of pieces, channels that end inside a block (the checks are those of test_gpu_conv_direct)."""
import numpy as np
import pytest

import test_gpu_conv_direct as layers

pytestmark = pytest.mark.gpu

CASES = [
    (1, 6, 6, 3, 2, 1, 1, True, 1, 1, 1, 1),       # six elements of filter
    (1, 9, 9, 1, 1, 2, 2, True, 1, 1, 1, 1),       # four
    (1, 9, 11, 1, 33, 7, 7, True, 1, 1, 1, 1),     # runs shorter than a piece
    (1, 12, 10, 2, 40, 5, 8, True, 1, 1, 1, 1),    # whole pieces only, ten and twenty of them
    (1, 14, 14, 3, 65, 7, 6, True, 2, 1, 1, 1),    # a run's last piece of two elements
    (2, 20, 16, 3, 64, 6, 7, True, 2, 2, 2, 1),    # eighteen pieces of the twenty-two that are kept
    (1, 70, 66, 3, 96, 7, 7, True, 1, 1, 1, 1),
]


@pytest.mark.parametrize("cfg", CASES)
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("start,infinite", [(0, False), (1, False), (0, True)])
def test_filters(oracle_port, cfg, dtype, start, infinite, monkeypatch):
    layers.test_few_channels(oracle_port, cfg, dtype, start, infinite, monkeypatch)


def test_more_workgroups_than_share_the_chip(oracle_port, monkeypatch):
    """fp32, ten groups of pieces, more than three workgroups a compute unit"""
    layers.test_few_channels(oracle_port, (100, 40, 40, 1, 64, 7, 7, True, 1, 1, 1, 1), np.float32, 0, False, monkeypatch)
