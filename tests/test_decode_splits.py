"""Into how many blocks single-token attention splits its keys (host code: no GPU)."""
import pytest

from alice_llm_amd.hip import ops


@pytest.mark.parametrize("n_seqs,kv_heads,context,head_dim,least,most", [
    # one and two kv heads of many keys: beyond some 40 splits combining them costs more than they save (two sequences of 8,192
    # keys of 2 heads of 256: 19 us with 24 or 32 splits, 23 with 62; eight of one head of 64: 10 us with 17 to 32, 13 with 11)
    (2, 2, 8192, 256, 16, 40), (4, 1, 8192, 256, 16, 40), (1, 1, 8192, 256, 16, 40), (8, 1, 8192, 64, 16, 40), (4, 1, 16384, 128, 16, 56),
    # the shapes of the 2B, 9B and 27B models: as ever
    (1, 4, 2560, 256, 15, 15), (8, 4, 2560, 256, 6, 6), (64, 4, 2560, 256, 1, 1), (2, 16, 5120, 128, 8, 8), (4, 8, 1024, 256, 6, 6),
    # fewer keys than a block's four waves take
    (1, 4, 100, 256, 1, 4), (1, 16, 1, 64, 1, 1)])
def test_splits_of_measured_shapes(n_seqs, kv_heads, context, head_dim, least, most):
    assert least <= ops.decode_splits(n_seqs, kv_heads, context, head_dim) <= most


def test_splits_are_bounded():
    for head_dim in (64, 128, 256):
        for kv_heads in (1, 2, 4, 16):
            for n_seqs in (1, 3, 16, 17, 64, 300):
                for context in (1, 31, 33, 500, 2048, 100000):
                    s = ops.decode_splits(n_seqs, kv_heads, context, head_dim)
                    assert 1 <= s <= max(1, min(64, 256 // (n_seqs * kv_heads), -(-context // 32)))
