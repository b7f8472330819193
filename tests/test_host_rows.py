"""The host entry point's page-locked rows, as far as they can be looked at without a device
(csrc/host_rows.h through tests/host/host_rows_test)."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host", "host_rows_test")


def test_steps_around_the_page_locked_rows():
    if not os.path.exists(BIN):
        pytest.fail("tests/host/host_rows_test is not built (run __graft_entry__.build())")
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    assert "later_piece_fails_and_is_waited_for" in r.stdout and "given_back_with_the_last" in r.stdout
