"""Norms in groups where a workgroup takes one group or some: sums at one, two and four quads of columns a lane and at sizes that none of them takes whole,
convolutions whose workgroups have more threads than columns or several turns of them, with one token and with many."""
import numpy as np
import pytest

from powerinfer_amd import lib as pl
from test_gpu_latent_ops import TYPES
from test_gpu_pufivik_ops import convolve, test_sums_and_norms_in_groups as sums_and_norms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("what", ["sum", "weighted experts", "norm only", "sum only"])
@pytest.mark.parametrize("T,cols,groups,ol", [(1, 256, 1, 0), (16, 4096, 16, 1), (3, 768, 1, 0), (2, 4096, 1, 1), (33, 2048, 8, 0), (2, 4608, 1, 0), (3, 4352, 1, 0), (1, 16384, 2, 0), (2, 10240, 1, 0), (1, 16384, 1, 0), (1, 17408, 1, 0)])
def test_sums_by_groups(t, T, cols, groups, ol, what):
    if not (ol and t == pl.F32):
        sums_and_norms(t, T, cols, groups, ol, what)


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("cols,groups,taps", [(520, 2, 4), (4096, 1, 4), (5120, 5, 3), (6144, 12, 2), (4, 1, 5), (9216, 3, 1)])
def test_convolutions_by_groups(t, cols, groups, taps):
    for runs in ([(2, [1, 1, 1, 1]), (0, [1, 1, 0, 1]), (1, [0, 1, 1, 1])], [(2, [37, 1, 2, 1]), (0, [1, 1, 1, 9]), (4, [2, 60, 0, 1])]):
        convolve(t, runs, cols, groups, taps, 0, np.random.default_rng(cols + taps), 4)
