"""The Toeplitz length rule over its whole range, without a GPU: every width from
243 to 4096 gets a length that has compile-time passes, no shorter than 2n - 1
and within 1/7 of the smallest even 2,3,5,7-smooth length."""

import ctypes as C
import os
import re

CSRC = os.path.join(os.path.dirname(__file__), "..", "tomocam_amd", "csrc")


def _plans():
    """Planned lengths as the sources list them."""
    with open(os.path.join(CSRC, "toeplitz_ct.h")) as f:
        plain = re.findall(r"PlainPlan(\d+) = TPlan<", f.read())
    with open(os.path.join(CSRC, "toeplitz_ct.hip")) as f:
        mixed = re.findall(r"using Plan(\d+) =", f.read())
    assert len(plain) == 23 and len(mixed) == 9
    return {int(v) for v in plain + mixed}


def _smooth(m):
    m += m % 2
    while True:
        r = m
        for p in (2, 3, 5, 7):
            while r % p == 0:
                r //= p
        if r == 1:
            return m
        m += 2


def test_every_width_has_a_plan():
    from tomocam_amd import _lib
    plans, m = _plans(), C.c_int()
    for n in range(243, 4097):
        _lib.call("tc_toeplitz_fft_length", n, C.byref(m))
        s = _smooth(2 * n - 1)
        assert m.value in plans, n
        assert 2 * n - 1 <= m.value <= s + s // 7


def test_every_plan_has_a_gpu_test():
    import test_gpu_toeplitz
    import test_gpu_toeplitz_plain as plain
    import test_gpu_toeplitz_widths as more
    listed = {M for _, _, M in plain.PLANS + plain.LARGE + more.WIDTHS}
    for m in test_gpu_toeplitz.test_toeplitz_sizes.pytestmark:
        if m.name == "parametrize":
            listed |= {M for _, _, M in m.args[1]}
    assert _plans() <= listed
