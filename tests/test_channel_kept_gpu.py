"""The channel decays' block kernel with its keys kept in LDS (heads of up to 128 in whole tiles of 16) and, just past that line, in the workspace."""
import pytest

from test_delta_blocks_gpu import test_delta_blocks_against_64_bits as against_64_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,D,Dv", [(2, 1, 48, 47), (3, 3, 112, 130), (2, 2, 128, 17), (2, 1, 144, 128), (1, 1, 256, 16)])
def test_kept_keys_against_64_bits(H, G, D, Dv):
    """Fewer tiles than fit, all of them, one more than fit; the bound over chains of up to 330 tokens is the imported test's."""
    against_64_bits(True, H, G, D, Dv, 0)
