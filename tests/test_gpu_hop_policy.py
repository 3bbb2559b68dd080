"""The reduced-precision hopping kernels with two waves per site and the operator
streamed past the caches: FP32 fields from 307 k sites per parity, FP32 spinors
with 16-bit links from 371 k, both to 524 k.  As, and with the bounds of, the test
of the kernels' other forms; 428400 sites leave a remainder in the last workgroup."""
import pytest

from test_gpu_hop_split import test_reduced_operators as operators

pytestmark = pytest.mark.gpu


def test_two_waves_streamed():
    operators((30, 28, 30, 34))
