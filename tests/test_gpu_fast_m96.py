"""GPU parity of the FAST scan compiled for 96 codebooks: subvectors of 8 (the
width fixed at compile time) and of 2 (the run-time width)."""

import pytest

from test_gpu_fast_shapes import test_fast_scan_shapes_against_oracle as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,M", [(768, 96), (192, 96)])
def test_96_codebooks(oracle, d, M):
    _check(oracle, d, M)
