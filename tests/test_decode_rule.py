"""Which calls go to the decode kernel (hbsa_fwd_decodes): by the longest q block there may be, not by the mean alone."""
import pytest

from hbsattn_amd import _lib


def _decodes(rows, hq, hk, qbs, k_lens, kbs=64, dtype=_lib.DTYPE_BF16):
    """``rows``: query lengths of the sequences; every sequence is cut into blocks of ``qbs``."""
    blocks = sum(-(-n // qbs) for n in rows)
    return _lib.load().hbsa_fwd_decodes(dtype, sum(rows), hq, hk, blocks, sum(-(-n // kbs) for n in k_lens), qbs, kbs)


@pytest.mark.parametrize("rows,hq,hk,qbs,expected", [
    ([1] * 32, 32, 8, 16, 1),              # decode steps
    ([1] * 32, 32, 8, 128, 1),             # in blocks of any size: one row each is all there can be
    ([1, 4, 2, 3] * 8, 32, 8, 16, 1),      # drafts: 64 entries at most
    ([1, 4, 2, 3] * 8, 32, 8, 64, 0),      # 49 rows at most for all that is known
    ([1] * 60 + [128], 32, 8, 16, 1),      # a chunk among decode steps: 16-row blocks of 64 entries ...
    ([1] * 60 + [128], 32, 8, 32, 0),      # ... 128
    ([1] * 60 + [128], 32, 8, 128, 0),     # ... 512
    ([1] * 60 + [128], 16, 16, 128, 0),    # ... 128
    ([1] * 60 + [64], 16, 2, 16, 0),       # 128
    ([5] * 8, 32, 8, 16, 0),               # 20 entries on average
])
def test_by_the_longest_block(rows, hq, hk, qbs, expected):
    assert _decodes(rows, hq, hk, qbs, [4000] * len(rows)) == expected
    assert _decodes(rows, hq, hk, qbs, [4000] * len(rows), dtype=_lib.DTYPE_F16) == expected
    for dtype in (_lib.DTYPE_F32, _lib.DTYPE_F32_STAGED16):
        assert _decodes(rows, hq, hk, qbs, [4000] * len(rows), dtype=dtype) == 0


@pytest.mark.parametrize("rows,k_lens,hk,kbs,expected", [
    ([2048] * 4, None, 4, 64, 1),            # 2048 items
    ([4096], None, 4, 64, 0),                # 1024 of long sequences
    ([4096], None, 4, 48, 1),                # k blocks smaller than the other kernel's tiles
    ([540] * 3, [4300] * 3, 1, 32, 0),       # ... but few items of many keys
    ([540] * 3, [4300] * 3, 4, 32, 1),
    ([160] * 8, [9000] * 8, 32, 64, 0),      # chunks
    ([32768], None, 8, 64, 1),
    ([32768], None, 16, 64, 0),              # more K and V than the caches hold
    ([300], None, 8, 64, 1),                 # short
    ([1000], None, 8, 64, 0),
    ([100] * 16, None, 2, 64, 1),            # short, as the rows missing in the last blocks tell
    ([16] * 32, [40000] * 32, 8, 64, 0),     # whole blocks of queries on long caches: no parts, too few items
])
def test_full_blocks(rows, k_lens, hk, kbs, expected):
    """16-row blocks, one q head per kv head: every prefill and training call has items of at most 16 entries."""
    assert _decodes(rows, hk, hk, 16, k_lens or rows, kbs) == expected


def test_sizes_that_make_no_call():
    lib = _lib.load()
    good = [_lib.DTYPE_BF16, 32, 32, 8, 32, 2000, 16, 64]
    assert lib.hbsa_fwd_decodes(*good) == 1
    for i in range(1, 8):
        assert lib.hbsa_fwd_decodes(*good[:i], 0, *good[i + 1:]) == 0
    assert lib.hbsa_fwd_decodes(_lib.DTYPE_BF16, 32, 30, 8, 32, 2000, 16, 64) == 0   # q heads no multiple of the kv heads
