"""The float32 prep's LDS overlays: L and A where the key tile was, the value columns staged 128 at a time (64 where the
query tile holds no more) in the other tile.  One token, whole and ragged chunks, stages with a remainder of 32 columns,
key widths in one pass and in several: the float64 oracle at the float32 rule's bar."""
import pytest

from oracle import gdr
from test_gpu_dropin import check_rule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 2, 128, 160), (1, 64, 2, 128, 32), (2, 65, 1, 160, 160), (1, 129, 2, 96, 160),
                                   (1, 70, 3, 256, 96), (1, 63, 2, 32, 96)])
def test_prep_stages(shape):
    print("case float32 prep", shape, flush=True)
    check_rule(gdr.harness_inputs(*shape, seed=5), 2e-4)
