"""The forward's split count (through its workspace): host only."""
import pytest

from chronicals_amd import _lib


@pytest.mark.parametrize("N", [1, 255, 256, 257, 700, 1500, 4096, 16384, 65536, 2 ** 21])
@pytest.mark.parametrize("V", [1, 256, 257, 5003, 50257, 151936])
def test_split_count_bounds(N, V):
    """Every row's lse: at least one round of workgroups where the tiles allow
    it, and never more splits than about 512 workgroups or min(32, 2048 / row
    tiles) per row tile; each has a slot of 256 rows of two fp32 partials."""
    gm, tn = -(-N // 256), -(-V // 256)
    most = min(max(-(-512 // gm), min(32, -(-2048 // gm))), tn)
    least = min(most, -(-256 // gm))
    slot = 256 * 8
    got = _lib.forward_workspace_bytes(N, 72, V, _lib.CCE_REDUCTION_MEAN)
    # what the workspace holds beside the partials: block sums, row losses, the column sums of W
    rest = 8 * -(-N // 4) + 4 * N + 4 * 72 * 65 + 16 * 256
    assert least * gm * slot <= got <= most * gm * slot + rest
