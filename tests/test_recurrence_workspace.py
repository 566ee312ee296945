"""What the recurrences by chunks ask for as scratch memory (host code: no GPU)."""
import pytest

from alice_llm_amd.hip import ops


@pytest.mark.parametrize("T,n_seqs,H,d,dv,delta", [(16384, 8, 16, 128, 128, 1), (8192, 1, 64, 128, 128, 1), (100000, 1, 64, 256, 256, 1),
                                                   (10 ** 6, 1, 64, 128, 64, 0), (300, 64, 16, 128, 128, 1)])
def test_the_workspace_is_bounded(T, n_seqs, H, d, dv, delta):
    need = lambda T: ops.library().alice_recurrence_chunks_workspace(T, n_seqs, H, 1, d, dv, delta)      # noqa: E731
    assert 0 < need(T) <= 1 << 26 and need(10 * T) <= 1 << 26
    assert need(16) <= need(300) <= need(T)
