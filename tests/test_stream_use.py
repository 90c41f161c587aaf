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


def test_one_shot_batches_share_no_lock():
    """A one-shot batch runs on buffers and streams of its own: it takes no
    lock over its work, so calls of several threads run side by side (when
    they end also depends on the hardware queues their streams are given)."""
    code = _code("capi.cpp")
    at = code.index("int pqp_permanent_batch_c128(")
    body = code[at: code.index("\n}\n", at)]
    assert "OneShotLease lease" in body
    assert "single_state" not in body and "lock_guard" not in body and "unique_lock" not in body
