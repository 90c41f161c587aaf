"""The library's streams are non-blocking: nothing orders them after the null
stream, so memory they use is cleared and copied on the streams themselves."""

import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _code(name):
    text = open(os.path.join(ROOT, "piquasso_amd", "csrc", name)).read()
    return re.sub(r"//[^\n]*", "", text)


@pytest.mark.parametrize("name", ["capi.cpp", "noalloc.hip"])
def test_no_clear_on_the_null_stream(name):
    assert not re.findall(r"\bhipMemset\w*\((?![^;]*[sS]tream)[^;]*;", _code(name))


def test_streams_are_created_once():
    """Every stream comes from ensure_stream, which leaves one that a failed
    call created to the next call."""
    code = _code("capi.cpp")
    assert len(re.findall(r"hipStreamCreate", code)) == 1
    assert re.search(r"int ensure_stream\(hipStream_t &stream\) \{\s*if \(!stream\)", code)
