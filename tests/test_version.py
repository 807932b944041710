"""The library answers with the version of the header that it was built from, which moves with the contracts."""
import os
import re

from fsa_hip import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_version_is_that_of_the_header():
    text = open(os.path.join(ROOT, "include", "fsa_hip.h")).read()
    version = int(re.search(r"#define FSA_HIP_VERSION (\d+)", text).group(1))
    assert _lib.load().fsa_version() == version >= 220
