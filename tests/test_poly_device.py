"""The device root finder's register form (poly_device.h, plain arithmetic that
also builds for the host) against its stack form: same roots, bit for bit, on
torus quartics, wide-ranging, degenerate and non-finite polynomials."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def poly_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("poly") / "poly_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", os.path.join(HERE, "poly_check.cpp"),
                           "-o", exe])
    return exe


# form, polynomials, whether roots and degenerate chains must be among them
@pytest.mark.parametrize("form,n,roots,degenerate", [(0, 200000, True, False), (1, 100000, True, False),
                                                     (2, 100000, True, True), (3, 100000, True, True),
                                                     (4, 50000, False, False)])
def test_register_form_equals_stack_form(poly_check, form, n, roots, degenerate):
    bad, deg, found = map(int, subprocess.check_output([poly_check, str(form), str(n)]).split())
    assert bad == 0
    assert not roots or found > 0
    assert not degenerate or deg > 0
