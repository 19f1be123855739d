"""The block map at the lines of its launches: items per side around one sort's threads and the
waves of it, and key-mask rows whose first active key comes late or never."""

import numpy as np
import pytest

from test_gpu_blockmap import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows, t", [(1, 1), (63, 5), (64, 5), (65, 5), (1, 8320), (511, 130),
                                     (512, 130), (513, 130), (1024, 3), (1025, 3)])
def test_order_item_counts(rows, t, device):
    rng = np.random.default_rng(rows + t)
    seg = np.sort(rng.integers(0, 4, (rows, t)), axis=1).astype(np.int32)
    mask = (rng.random((rows, t)) < 0.9).astype(np.int32)
    _check(0, mask, seg, t, t, device)


@pytest.mark.parametrize("s", [1, 511, 512, 513, 1300, 2560, 2561, 4700])
def test_key_mask_rows_with_late_or_no_keys(s, device):
    rng = np.random.default_rng(s)
    mask = np.zeros((6, s), np.int32)
    mask[0, s - 1] = 1
    mask[1, s // 2] = -3
    mask[3] = rng.integers(0, 2, s)
    mask[4] = 1
    mask[5, : s // 3] = 7
    _check(2, mask, None, 300, s, device)
