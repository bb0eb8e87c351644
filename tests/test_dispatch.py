"""Which kernel a call runs, by the rules the entry points apply (host code, no GPU: the CU count is an argument)."""
import ctypes

import pytest

CUS = 256


def attention_plan(sq, sk, h, raw=False, tail=True, cus=CUS):
    """(queries per workgroup, queries quantized by the main kernel, workgroups run as two key halves)"""
    from rapid_h3 import _native as nat
    p = (ctypes.c_int64 * 3)()
    nat.call("rh3_attention_plan", sq, sk, h, int(raw), int(tail), cus, p)
    return tuple(p)


@pytest.mark.parametrize("sq,sk,h,npair", [(5583, 5583, 24, 104), (2600, 5583, 49, 87)])
def test_attention_plan_counts_the_split_only_where_it_runs(monkeypatch, sq, sk, h, npair):
    """A half-empty last round of 384-query workgroups is half as long only when its key halves can run: without room
    for the partials, or with RH3_ATTN_SPLIT=0, it costs a whole one and the finer 128-query grid is the faster."""
    monkeypatch.delenv("RH3_ATTN_SPLIT", raising=False)
    assert attention_plan(sq, sk, h) == (384, 0, npair)
    assert attention_plan(sq, sk, h, tail=False) == (128, 0, 0)
    assert attention_plan(sq, sk, h, raw=True, tail=False) == (128, 1, 0)
    monkeypatch.setenv("RH3_ATTN_SPLIT", "0")
    assert attention_plan(sq, sk, h) == (128, 0, 0)
    monkeypatch.setenv("RH3_ATTN_SPLIT", "1")
    assert attention_plan(sq, sk, h) == (384, 0, npair)


def test_attention_plan_short_and_long_items():
    assert attention_plan(1024, 1024, 24) == (128, 0, 0)
    assert attention_plan(2816, 2816, 24) == (384, 0, 0)
    assert attention_plan(2816, 2816, 24, raw=True) == (128, 1, 0)      # it saves the pre-pass over the queries
    assert attention_plan(1024, 65536, 24)[0] == 128
    assert attention_plan(1024, 65537, 24)[0] == 384                    # past the 128-query kernel's scale table
