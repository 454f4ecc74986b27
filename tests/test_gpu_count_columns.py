"""Per-class bit counts at the edges of the column kernel: every piece width a row length allows, one column, the last block
of columns partly empty, classes of fewer rows than a wavefront has row phases, the row counts around one and two steps of
eight rows per phase, and classes beyond the counters' range (row slices)."""
import numpy as np
import pytest
import torch

from convlogic_amd.hip import difflogic_hip
from oracle import convlogic_oracle as O
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,words", [(64, 1), (64, 3), (64, 64), (64, 65), (64, 130), (32, 1), (32, 7), (32, 129), (16, 5), (8, 1), (8, 77)])
@pytest.mark.parametrize("class_rows,k", [(1, 3), (7, 2), (63, 10), (64, 1), (65, 2), (513, 2), (1100, 3)])
def test_counts_at_the_edges_of_the_column_kernel(bits, words, class_rows, k):
    rng = np.random.default_rng(bits * 1000 + words + class_rows)
    dtype = {8: np.int8, 16: np.int16, 32: np.int32, 64: np.int64}[bits]
    info = np.iinfo(dtype)
    x = rng.integers(info.min, info.max, size=(class_rows * k, words), dtype=dtype, endpoint=True)
    pad = int(rng.integers(0, bits)) if words > 1 else 0
    got = difflogic_hip.groupbitsum(torch.from_numpy(x).to(DEV), pad, k)
    assert np.array_equal(got.cpu().numpy(), O.group_bit_sum(x, pad, k))


@pytest.mark.parametrize("bits,words", [(64, 2), (32, 3)])
def test_counts_of_classes_beyond_the_counter_range(bits, words):
    dtype = {32: np.int32, 64: np.int64}[bits]
    x = np.full((2 * 16400, words), -1, dtype=dtype)                   # every bit set: the largest count of every position
    x[16400:16411] = 0
    got = difflogic_hip.groupbitsum(torch.from_numpy(x).to(DEV), 1, 2).cpu().numpy()
    assert got.shape == (words * bits - 1, 2) and (got[:, 0] == 16400).all() and (got[:, 1] == 16400 - 11).all()
