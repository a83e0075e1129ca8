"""Device memory is never cleared on the null stream: hipMemset returns before
it has run, and the contexts' streams are created with hipStreamNonBlocking, so
nothing orders such a clear before what is put there on a context's stream next.
Read from the sources: a clear that lands late leaves no error to test for."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sagesim_amd", "csrc")


def _code(name):
    with open(os.path.join(CSRC, name)) as f:
        text = f.read()
    return re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)


@pytest.mark.parametrize("name", sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".h"))))
def test_no_clear_on_the_null_stream(name):
    calls = re.findall(r"\bhipMemset(?:D8|D16|D32|2D|3D)?\s*\([^;]*;", _code(name))
    assert not calls, calls
