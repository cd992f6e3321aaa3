"""Host checks of the rate-control code shared by the host library and the GPU (rc_shared.h)."""
import ctypes as C
import os

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "librc_host.so")


@pytest.mark.parametrize("passes", [0, 1, 3, 4, 5, 22, 61, 64])
def test_hull_copies_no_unset_pass(passes):
    """The hull takes a block's passes in groups; those past the block's last hold a value."""
    if not os.path.exists(LIB):
        pytest.skip("tests/native/librc_host.so not built (make -C tests/native)")
    assert C.CDLL(LIB).rc_pass_entries_unset(passes) == 0
