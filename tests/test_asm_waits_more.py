"""The wait-count check of tests/asm_waits.py over the sources that
tests/test_asm_waits.py does not name; with INQX_ASM_CHECK=1."""
import os

import pytest

from tests.test_asm_waits import test_library_kernels as check_source


@pytest.mark.skipif(os.environ.get("INQX_ASM_CHECK") != "1", reason="compiles the sources; set INQX_ASM_CHECK=1")
@pytest.mark.parametrize("src", ["density", "small_grid"])
def test_further_sources(src, tmp_path):
    check_source(src, tmp_path)
