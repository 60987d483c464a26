"""psy_ctx_reset_trace_form: the main pass's form as on a new context."""
import ctypes as C

import pytest

from psychopath_cpp_amd import abi, gpu
from tests.cpu_build import hostbuild


@pytest.mark.parametrize("steps", [["mode"], ["continuation"], ["mode", "continuation"]])
def test_reset_gives_the_choice_back(steps):
    new = hostbuild.trace_form([])
    assert hostbuild.trace_form(steps) != new
    assert hostbuild.trace_form(steps + ["reset"]) == new


def test_reset_refuses_no_context():
    assert gpu.lib().psy_ctx_reset_trace_form(C.c_void_p()) == abi.PSY_ERR_INVALID
