"""dsx_workspace_bytes: what it answers is enough for any smaller number of pairs and any number of Gaussians."""
import pytest

from ds_splat_amd import _native


@pytest.mark.parametrize("W,H,bins", [(320, 320, 1), (640, 400, 1), (640, 640, 1), (1600, 1120, 2), (3840, 2160, 0), (64, 64, 0)])
def test_a_workspace_serves_fewer_pairs(W, H, bins):
    lib = _native.load()
    at = sorted({0, 1} | {max(0, k + d) for k in [items << 18 for items in range(1, 14)] + [3_500_000, 8_000_000, 12_000_000, 50_000_000]
                          for d in (-100_000, -1, 0, 1, 100_000)})
    sizes = [lib.dsx_workspace_bytes(0, k, W, H, bins) for k in at]
    assert sizes == sorted(sizes) and sizes[-1] < 9.1 * at[-1] + (1 << 20)
    for n in (1, 131_072, 131_073, 1 << 30):
        assert [lib.dsx_workspace_bytes(n, k, W, H, bins) for k in at] == sizes
