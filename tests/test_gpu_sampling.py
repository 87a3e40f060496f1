"""The sample streams at sample indices below, across and above the first
digit group of the Halton dimensions (243 samples in base 3, 125 in base 5):
a few pixels rendered at that many samples match the oracle's, whose sequence
takes every digit group of every sample."""

import pytest

from psychopath_amd import scenes
from tests.test_gpu_render import check_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spp", [1, 124, 126, 244, 1000])
def test_sample_counts_match_oracle(spp):
    check_parity(scenes.cornell_box(7, 5, spp, 2, 3), f"cornell 7x5x{spp}")
