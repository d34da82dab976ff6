"""The batched int8 kernels' workgroup tiles (csrc/int8.hip, chosen by
csrc/int8.c) at their edges, each forced, bit for bit against the oracle's
int8 lane: rows and tokens on both sides of 32, 64, 96 and 128, one to three
super-blocks, and token counts whose remainder past whole groups of four
takes the plain epilogue in one lane, one tile or everywhere.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import mynah_amd
    mynah_amd.check(mynah_amd.lib.mynah_hip_init(0), "init")
    return mynah_amd


@pytest.mark.parametrize("rows,cols,tokens", [
    (1, 256, 2), (31, 512, 3), (33, 256, 5), (64, 768, 32), (65, 512, 33), (95, 256, 64),
    (97, 512, 127), (128, 256, 128), (130, 768, 131), (200, 512, 213)])
@pytest.mark.parametrize("tile", ["0", "1", "2", "3", None])
@pytest.mark.parametrize("qtype", [12, 13])
def test_tiles_against_oracle(M, monkeypatch, qtype, tile, rows, cols, tokens):
    if tile is not None:
        monkeypatch.setenv("MYNAH_INT8_TILE", tile)
    w = M.synth_blocks(qtype, rows + tokens, rows, cols)
    x = M.synth_normal(cols, tokens * cols)
    M.set_int8(M.INT8_BATCHED)
    try:
        got = M.matmat(qtype, w, rows, cols, x, tokens)
    finally:
        M.set_int8(M.INT8_OFF)
    ref = np.empty(tokens * rows, np.float32)
    fn = O.orc.orc_q4k_matmat_int8 if qtype == 12 else O.orc.orc_q5k_matmat_int8
    assert fn(O.ptr(w), rows, cols, O.ptr(x), O.ptr(ref), tokens) == 0
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
