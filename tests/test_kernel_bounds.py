"""How far kernels read, computed on the host by the code that the kernels themselves use: what lies behind a tensor may not be mapped."""
import pytest


@pytest.mark.parametrize("D", [32, 128, 192, 320, 576])
def test_window_decode_loads_q_of_heads_that_there_are(D):
    """Decode attention's workgroups hold one or two chunks of 16 heads: also the waves without heads of their own (an odd number of
    chunks, 33, 40 or 80 heads of a wide row) load rows of q that belong to their sequence, and every head is loaded."""
    from llm_weighted_consensus_amd.ops import res32

    for G in (1, 2, 5):
        for Hg in range(1, 130):
            assert res32.kernels().window_attn_decode_heads(G * Hg, G, D) == (0, G * Hg - 1), (G, Hg)
