"""The admission estimate of a scene's blocks is its bounding box in blocks plus the +1
shell, whatever the cloud's length (around the 64 rows reduced at once), width, order and
type."""
import numpy as np
import pytest

from slosh_amd import scenes


@pytest.mark.parametrize("n", [0, 1, 3, 63, 64, 65, 128, 1000])
@pytest.mark.parametrize("width", [3, 4])
def test_estimate_is_the_box_in_blocks(n, width):
    pos = np.random.RandomState(n).uniform(-3.0, 3.0, (n, width))
    for a in (pos, pos.astype(np.float32), np.asfortranarray(pos), pos[::-1]):
        want = 0
        if n:
            h = 4.0 * 0.01
            want = int(np.prod([np.floor(a[:, i].max() / h) + 2 - np.floor(a[:, i].min() / h) + 2 for i in range(3)]))
        assert scenes.estimate_blocks(a, 0.01) == want
