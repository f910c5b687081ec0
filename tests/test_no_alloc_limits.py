"""tm_launch_noalloc's layout check, which comes before any GPU call: a program whose exact words and 8 control words
filled the array fits it with its 4,160 control words, and a byte more is refused."""
import ctypes

import pytest

from tallymap_amd.backend import compile as Cm

LIMIT, CTL = 32 << 20, 4160 * 4


@pytest.mark.parametrize("words, over", [(LIMIT - 256, 0), (LIMIT - 256, 225), (LIMIT - 300, 0), (LIMIT, 0),
                                         (LIMIT + 1, 0)])
def test_layout_limit(words, over):
    lib = Cm.lib()
    sl, nb = (ctypes.c_int * 2)(0, 1), (ctypes.c_longlong * 2)(words, CTL + over)
    bufs = (ctypes.c_void_p * 2)()
    rc = lib.tm_launch_noalloc(ctypes.c_longlong(-12345), None, bufs, 2, sl, nb, 2, 0, 0, 0, 256)
    assert rc != 0                      # (no such program, or no GPU: nothing runs in any case)
    at = -(-words // 256) * 256
    refused = words > LIMIT or at + 32 + over > LIMIT        # (with 8 control words)
    assert (b"no-alloc array" in lib.tm_last_error()) == refused
