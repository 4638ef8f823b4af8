"""The LDS-DMA protocol (M0 written by SALU one wait state before each copy, no
freshly written SGPR base) on the compiled fp32-mode triangle attention: its
attention core and its output linear stage their tiles by LDS DMA too."""

from pathlib import Path

import pytest
from test_lds_dma_protocol import HIPCC
from test_lds_dma_protocol import test_compiled_lds_dmas_follow_the_protocol as check

pytestmark = pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")


def test_fp32_attention_lds_dmas_follow_the_protocol(tmp_path):
    check("triattn_fp32", tmp_path)
