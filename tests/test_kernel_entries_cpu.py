"""What the kernel library's entry points refuse before they touch a device, in a process of its own: a crash ends that one."""
import subprocess
import sys

import pytest

from easy_gpt.cpp_amd.csrc import build

UNSUPPORTED_SIZE = 2
# One request of 2 heads of 64 on 1, one query token.  (No entry point gets as far as reading from the address.)
CALLS = """
import ctypes
lib = ctypes.CDLL({path!r})
p, ps, f = ctypes.c_void_p(4096), {page_size}, ctypes.c_float
none = ctypes.c_void_p(None)
print(lib.egpt_paged_attention_decode(p, p, p, p, p, p, p, 1, p, p, 1, 2, 1, 64, ps, f(1), 0, 1, 4, 1, 1, none),
      lib.egpt_attention_decode_fused(p, 1, none, 0, 0, f(0), none, p, p, p, p, p, p, p, p, 1, p, p, 1, 2, 1, 64, ps, f(1), 0, 1, 4, 1, 1, none),
      lib.egpt_attention_decode_ranged(p, 1, none, 0, 0, f(0), none, p, p, p, p, p, p, p, p, 1, p, p, 1, 2, 1, 64, ps, f(1), 0, p, 4, none),
      lib.egpt_paged_attention_mfma(p, p, p, p, p, p, p, 1, p, p, p, 1, 1, 2, 1, 64, ps, f(1), 0, 1, 16, 1, none))
"""


@pytest.mark.parametrize("page_size", [0, -16, 8, 24])
def test_attention_refuses_pages_that_are_no_multiple_of_sixteen_tokens(page_size):
    code = CALLS.format(path=build.ensure_built(), page_size=page_size)
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=110)
    assert p.returncode == 0, (p.returncode, p.stderr[-500:])
    assert p.stdout.split() == [str(UNSUPPORTED_SIZE)] * 4
