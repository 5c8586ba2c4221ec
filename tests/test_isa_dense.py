"""The ISA checks of tests/test_isa.py on the dense weights' kernels (CPU only)."""
import os
import subprocess

import pytest

from test_isa import CSRC, FLAGS, _hipcc, lds_read_hazards, mfma_result_hazards


def test_dense_lds_reads_and_mfma_results(tmp_path):
    hipcc = _hipcc()
    if not hipcc:
        pytest.skip("hipcc not available")
    path = str(tmp_path / "dense.s")
    subprocess.run([hipcc, *FLAGS, os.path.join(CSRC, "dense.hip"), "-o", path], check=True,
                   capture_output=True)
    text = open(path).read()
    assert lds_read_hazards(text) == []
    assert mfma_result_hazards(text) == []
