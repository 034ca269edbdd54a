"""Which prefill passes may be in flight together: those of one parity follow each other on a stream, so every even one's memory must lie apart from every odd one's."""
import pytest

from rtp_llm_amd import _C

A, B, D = 0x100000, 0x200000, 0x300000        # workspaces of 64 KB
VOCAB, SEQS = 1000, 3


def _apart(workspaces, logits=None):
    passes = (_C.PrefillPass * len(workspaces))()
    for i, (p, ws) in enumerate(zip(passes, workspaces)):
        p.workspace, p.workspace_bytes, p.nseq, p.logits_out = ws, 0x10000, SEQS, logits[i] if logits else None
    return _C.lib().mi355_prefill_passes_apart(passes, len(workspaces), VOCAB)


@pytest.mark.parametrize("workspaces,apart", [
    ([A], 1), ([A, B], 1), ([A, B, A, B, A], 1), ([A, A], 0), ([A, B, D], 1), ([A, B, D, B], 1),
    ([A, B, D, A], 0),                         # the fourth runs behind the second, which does not wait for the first's end
    ([A, B, D, B, D, A], 0), ([A, B, A, D, B], 0),
    ([A, A + 0x10000], 1), ([A, A + 0xFFFF], 0), ([A + 0xFFFF, A], 0),
])
def test_workspaces(workspaces, apart):
    assert _apart(workspaces) == apart


def test_logits():
    n = 4 * VOCAB * SEQS
    assert _apart([A, B, A, B], [D, D + n, D, None]) == 1
    assert _apart([A, B, A, B], [D, D + n - 4, None, None]) == 0
    assert _apart([A, B, A, B], [D, None, None, D]) == 0
