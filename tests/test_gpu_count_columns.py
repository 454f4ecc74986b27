"""Per-class bit counts at the edges of the column kernel: every piece width a row length allows, one column, the last block
of columns partly empty, classes of fewer rows than a wavefront has row phases, the row counts around one and two steps of
eight rows per phase, and classes beyond the counters' range (row slices)."""
import numpy as np
import pytest
import torch

from convlogic_amd.hip import difflogic_hip
from oracle import convlogic_oracle as O
from tests.gpu_util import DEV, set_knobs

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


# Few rows per class take a wavefront per class and 8 bytes of a row: at the ends of its range, columns that are partly behind the row,
# more (class, column) pairs than fill the GPU, and the column kernel at the same sizes (the knob takes it).
@pytest.mark.parametrize("bits,words", [(64, 1), (64, 9), (64, 63), (32, 1), (32, 15), (16, 5), (8, 1), (8, 77), (8, 1251)])
@pytest.mark.parametrize("class_rows,k", [(1, 700), (8, 3), (9, 100), (24, 70), (25, 70), (96, 2), (97, 2), (128, 3), (256, 2)])
def test_counts_of_classes_of_few_rows(bits, words, class_rows, k, monkeypatch):
    torch.manual_seed(bits + words + class_rows)
    x = torch.randint(-128, 128, (class_rows * k, words * bits // 8), dtype=torch.int8).view({8: torch.int8, 16: torch.int16, 32: torch.int32, 64: torch.int64}[bits])
    pad = int(torch.randint(0, bits, (1,))) if words > 1 else 0
    want = O.group_bit_sum(x.numpy(), pad, k)
    for slices in (None, "1"):
        set_knobs(monkeypatch, CLG_GSUM_SLICES=slices)
        assert np.array_equal(difflogic_hip.groupbitsum(x.to(DEV), pad, k).cpu().numpy(), want)
