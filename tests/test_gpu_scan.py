"""taco_hip_device_exclusive_scan against numpy: sizes around a thread's 16
counts, a tile of 4096 and the 2048 tiles up to which every workgroup adds up
the tiles before its own, and totals on both sides of the int32 range."""
import numpy as np
import pytest
import torch

from taco_amd import _lib

pytestmark = pytest.mark.gpu
TILE = 4096
DIRECT = 2048 * TILE
INT_MAX = (1 << 31) - 1


def _scan(counts, shift=0):
    """pos of the counts, the arrays `shift` words into their buffers."""
    m = len(counts)
    c = torch.zeros(m + shift, dtype=torch.int32, device="cuda")[shift:]
    c.copy_(torch.from_numpy(counts))
    pos = torch.full((m + 2 + shift,), -7, dtype=torch.int32, device="cuda")[shift:]
    _lib.check(_lib.lib().taco_hip_device_exclusive_scan(c.data_ptr(), m, pos.data_ptr()))
    got = pos.cpu().numpy()
    assert got[m + 1] == -7
    return got[:m + 1]


@pytest.mark.parametrize("m", [0, 1, 15, 16, 17, 255, 256, 4095, 4096, 4097, 70001, DIRECT - 1,
                               DIRECT, DIRECT + 1, DIRECT + 3 * TILE + 5, 20_000_003])
@pytest.mark.parametrize("shift", [0, 1])
def test_against_cumsum(m, shift):
    counts = np.random.default_rng(m).integers(0, 100, m, dtype=np.int32)
    expect = np.concatenate([[0], np.cumsum(counts, dtype=np.int64)])
    assert expect[-1] <= INT_MAX
    assert np.array_equal(_scan(counts, shift), expect)


@pytest.mark.parametrize("m", [1, 5 * TILE, DIRECT + 5 * TILE + 9], ids=["one", "direct", "large"])
@pytest.mark.parametrize("where", ["first", "middle", "last", "spread"])
def test_int32_range(m, where):
    counts = np.zeros(m, np.int32)
    if where == "spread":
        counts[:] = INT_MAX // m
        counts[m // 3] += INT_MAX - int(counts.sum(dtype=np.int64))
    else:
        counts[{"first": 0, "middle": m // 2, "last": m - 1}[where]] = INT_MAX
    assert np.array_equal(_scan(counts), np.concatenate([[0], np.cumsum(counts, dtype=np.int64)]))
    # One more, in the first, a middle and the last count in turn.
    for at in {0, m // 2, m - 1}:
        if counts[at] == INT_MAX:
            continue
        counts[at] += 1
        with pytest.raises(_lib.TacoHipError):
            _scan(counts)
        counts[at] -= 1
