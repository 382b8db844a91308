"""The C interface's version: one number in the header, the library and the
binding, which refuses a library of another."""
import os
import re

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "pysweep_hip.h")


def test_header_library_and_binding_agree():
    from pysweep_amd import hip
    declared = int(re.search(r"^#define PS_VERSION (\d+)$", open(HEADER).read(), re.M).group(1))
    # 6 had shorter plans (no chain, full, full_rows, band_step) and no ps_write
    assert declared >= 7
    assert hip.version() == declared == hip.ABI_VERSION


@pytest.mark.parametrize("version", [6, 8])
def test_another_version_is_refused(version):
    from pysweep_amd import hip
    with pytest.raises(ImportError, match=f"version {version}.*build"):
        hip.check_abi(version)
