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


@pytest.mark.parametrize("planes", [1, 4, 112])
def test_gemm8p_reads_block_scales_of_rows_that_there_are(planes):
    """Dense fp8 products of an A with block scales [planes, rows, 4]: row blocks are views of the scales, and no tile of any block may
    load from behind the tensor (the last rows' tile: 256 rows whatever is left), while each row's scales lie in what it may load."""
    from llm_weighted_consensus_amd import ops

    k, size = ops.kernels(), 4
    for rows, blocks in ((1200, [(0, 1200)]), (1200, [(0, 512), (512, 1024), (1024, 1200)]), (1025, [(0, 1024), (1024, 1025)]),
                         (149761, [(0, 149760), (149760, 149761)])):
        for r0, r1 in blocks:
            for tile in (192, 224, 256):
                for m0 in {0, (r1 - r0 - 1) // tile * tile}:
                    span = k.gemm8p_mx_bytes(planes, rows, r1 - r0, m0)
                    assert (r0 + m0) * size + span <= planes * rows * size, (rows, r0, r1, m0)
                    assert span >= ((planes - 1) * rows + min(tile, r1 - r0 - m0)) * size, (rows, r0, r1, m0)
