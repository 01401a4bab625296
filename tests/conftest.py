import os
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP path)")
    config.addinivalue_line("markers", "slow: long-running case")


def pytest_report_header(config):
    return [f"sonic-amd repo root: {ROOT}"]


# Tests that measure against the reference's own translation units, built
# with and without FMA contraction from its sources (oracle/Makefile).
NEEDS_REFERENCE_BUILDS = {"test_batch_teno5_at_300_steps_within_the_references_own_spread"}


def pytest_collection_modifyitems(items):
    from oracle import bind
    if bind.ref_available() and bind.ref_fma_available():
        return
    for item in items:
        if item.name in NEEDS_REFERENCE_BUILDS:
            item.add_marker(pytest.mark.skip(reason="reference harness not built"))
