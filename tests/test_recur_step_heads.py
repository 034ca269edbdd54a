"""Which heads the recurrence step of few rows takes: what its launch has an instance for, all other heads walk."""
from rtp_llm_amd import hybrid_ops as hops


def test_heads_with_an_instance():
    for vdim in range(1, 300):
        for dim in range(1, 300):
            one = vdim % 4 == 0 and vdim <= 256 and dim <= 256 and dim * vdim <= 32768
            fits = one and -(-dim // (256 // (vdim // 4))) <= 36             # key rows of a thread that holds four columns
            assert hops.recur_step_supported(dim, vdim) is fits, (dim, vdim)
