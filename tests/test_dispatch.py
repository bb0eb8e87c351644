"""Which kernel a call runs, by the rules the entry points apply (host code, no GPU: the CU count is an argument)."""
import ctypes

import pytest

from conftest import GEMM_COUNTED, GEMM_SHARES, GEMM_SINGLE, GEMM_SMALL, gemm_plan
from conftest import attention_plan as device_plan


def attention_plan(*args, full=False, **kw):
    return device_plan(*args, cus=256, **kw)[:4 if full else 3]


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


def test_attention_plan_out_over_the_queries():
    """The main kernel quantizes the queries itself only where no other workgroup's out rows can lie on them."""
    s, h = 1024, 24
    base, row = 1 << 40, 2 * 128
    q = (base, h * 128, 128)                                 # [S, H, 128]
    end = base + s * h * row

    def raw(out, q=q):
        return attention_plan(s, 512, h, q=q, out=out)[1]
    assert raw((base, h * 128, 128)) == 1                    # in place
    assert raw((base, 128, s * 128)) == 0                    # head-major over the same storage
    assert raw((base + row, h * 128, 128)) == 0              # one head on
    assert raw((end - row, h * 128, 128)) == 0               # over the last head of the last token
    assert raw((end, h * 128, 128)) == 1                     # right behind q, and right before it
    assert raw((base - s * h * row, 128, s * 128)) == 1
    assert raw((base - s * h * row + row, 128, s * 128)) == 0
    assert raw((end - row, -h * 128, -128)) == 0             # rows and heads backwards over q
    assert raw((end + (s * h - 1) * row, -h * 128, -128)) == 1
    fused = (base, 3 * h * 128, 128)                         # q of a [S, 3, H, 128] buffer, out in its v part
    assert raw((base + 2 * h * row, 3 * h * 128, 128), q=fused) == 0
    # the plan without it is that of a call whose pre-pass quantizes the queries
    assert attention_plan(s, 512, h, q=q, out=(base, 128, s * 128)) == attention_plan(s, 512, h)


def test_attention_grids_stay_below_the_launch_limit():
    """A one-dimensional grid holds 2^24 - 1 workgroups of 256 threads: past that the query kernel, or the merged
    pre-pass, of the other form is taken, and the production pre-passes name the limit before any launch."""
    from rapid_h3 import _native as nat
    h = 300
    most = ((1 << 24) - 1) // h                               # 128-query workgroups per head
    assert attention_plan(most * 128, 64, h) == (128, 0, 0)
    assert attention_plan((most + 1) * 128, 64, h)[0] == 384
    assert attention_plan((most - 3) * 128, 64, h, full=True)[3] == 1   # and a chunk of K statistics, two 64-key V slabs
    assert attention_plan(most * 128, 64, h, full=True)[3] == 0
    assert attention_plan(4096, 4096, 24, full=True)[3] == 1
    assert attention_plan(4096, 4097, 24, full=True)[3] == 0
    fake = ctypes.c_void_p(0x1000)                            # never dereferenced: refused first
    big = ctypes.c_int64(1 << 62)
    s, h = 4_000_000, 200                                     # S H (1/64 + 1/128) = 18.75 M workgroups
    qkv = [fake, 128, 128] * 3
    tail = [1, 1, 1, fake, 128, 128, fake, big, None]
    for name, mid in (("rh3_int8_attention_u8", [None, 0, None, None, 1e-5, 0.1, 0, 0.0]),
                      ("rh3_int8_attention_bk", [0.1])):
        st = getattr(nat.lib(), name)(*qkv, s, s, h, *mid, *tail)
        assert st == 1 and "beyond the grid limit" in nat.last_error(), (name, nat.last_error())


@pytest.mark.parametrize("m,n,k,plan", [
    (77, 9216, 3072, (128, 64, 0, GEMM_SMALL)), (512, 6144, 3072, (128, 128, 0, GEMM_SMALL)),
    (700, 784, 1024, (128, 64, 0, GEMM_SMALL)), (129, 16528, 64, (256, 128, 0, GEMM_SMALL)),
    (1029, 15376, 512, (256, 192, 0, GEMM_SMALL)),
    (1029, 15376, 1024, (128, 64, 1024, GEMM_SHARES)),           # whole rounds, then the last rows
    (4096, 3072, 3072, (256, 256, 4096, GEMM_SHARES)),
    (5300, 6096, 512, (256, 256, 5300, GEMM_SHARES)), (5300, 6096, 320, (256, 256, 5300, GEMM_SINGLE)),
    (4100, 15616, 512, (256, 256, 4100, GEMM_COUNTED)),
    (9000, 8200, 256, (256, 256, 9000, GEMM_SINGLE)),            # K below 512
    (145152, 9216, 3072, (256, 256, 145152, GEMM_COUNTED))])
def test_gemm_plan(m, n, k, plan):
    assert gemm_plan(m, n, k, cus=256) == plan


def test_gemm_counters_from_four_rounds_on():
    assert gemm_plan(4 * 256 * 256, 256, 512, cus=256)[3] == GEMM_COUNTED
    assert gemm_plan(4 * 256 * 256 - 256, 256, 512, cus=256)[3] == GEMM_SHARES
