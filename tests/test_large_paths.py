"""What large calls take (slabs of 65536 elements or as _SLAB says, a lane per decoded block, the auxiliary
stream, scans in several launches, uploads of their own), at the sizes of the other tests: CRX_LARGE_PATHS
makes calls of every size take it, and the tests below are those files' own."""

import pytest

from test_api import *  # noqa: F401,F403
from test_call_sizes import (test_blocks_of_long_codes, test_blocks_of_long_remainders,  # noqa: F401
                             test_decoder_by_number_of_blocks)
from test_full_sizes import (test_small4_every_header_byte_every_block_boundary_and_10k_payload_flips,  # noqa: F401
                             test_small4_widened_flips_with_small_slabs)
from test_parity import *  # noqa: F401,F403

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _large_paths(monkeypatch):
    monkeypatch.setenv("CRX_LARGE_PATHS", "1")
