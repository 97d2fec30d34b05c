"""What the BatchNorm training entry points refuse, by their own checks ahead of any launch (no GPU
needed: the pointers are never read)."""

import pytest

import oxide_hip as ox

BASE = 0x7F0000000000


# channels kept whole, by slices, one plane of 64 values, eight units per thread
@pytest.mark.parametrize("shape", [(8, 64, 20 * 20), (64, 128, 56 * 56), (2, 3, 64),
                                   (32, 128, 32 * 32)])
def test_forward_refuses_a_workspace_inside_the_input(shape):
    n, c, hw = shape
    size = ox.batch_norm_workspace_size(n, c, hw)
    far = [BASE + (i + 2) * (1 << 40) for i in range(8)]
    status = ox.lib().oxh_batch_norm_forward_train(
        None, n, c, hw, 0.1, 1e-5, BASE, *far[:6], far[6], BASE + 4 * (n * c * hw // 2 // 4 * 4),
        size)
    with pytest.raises(ox.OxideError, match="workspace overlaps the input"):
        ox.check(status)
