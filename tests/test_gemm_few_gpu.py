"""The MFMA GEMM's kernels for at most 32 tokens (four columns of one 16-token
group an instruction; csrc/gemm_mfma.hip), bit for bit against the VALU kernels
of csrc/gemm_exact.hip, in both orders: tokens around the 16-token groups and
the line at 32, rows around the wave and the tile, one to ten super-blocks,
with and without splits through memory; any bit pattern and non-finite
activations.
"""
import numpy as np
import pytest

from test_gemm_tiles_gpu import M, product, same  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 2, 15, 16, 17, 31, 32, 33])
@pytest.mark.parametrize("rows,units", [(1, 1), (17, 2), (63, 3), (200, 10)])
@pytest.mark.parametrize("mv", [False, True])
@pytest.mark.parametrize("qtype", [12, 13, 14, 8])
def test_few_tokens(M, monkeypatch, qtype, mv, rows, units, tokens):  # noqa: F811
    cols = 256 * units
    rng = np.random.default_rng(tokens)
    odd = M.synth_normal(3, tokens * cols).copy()
    odd[[5, 7, cols // 2, cols - 1]] = np.inf, 3e37, 1e-41, np.nan
    for w, x in ((M.synth_blocks(qtype, rows, rows, cols), M.synth_normal(units, tokens * cols)),
                 (rng.integers(0, 256, rows * M.row_bytes(qtype, cols), dtype=np.uint8), odd)):
        res = M.synth_normal(tokens, tokens * rows) if mv else None
        ref = product(M, monkeypatch, {"MYNAH_GEMM_MFMA": "0"}, mv, qtype, w, rows, cols, x,
                      tokens, res)
        for env in ({}, {"MYNAH_GEMM_SPLIT": "0"}, {"MYNAH_GEMM_SPLIT": "3"}):
            got = product(M, monkeypatch, env, mv, qtype, w, rows, cols, x, tokens, res)
            assert same(got, ref), env


@pytest.mark.parametrize("rows,cols,tokens", [(4096, 2560, 65), (4095, 2560, 80), (2048, 2048, 270),
                                              (2560, 9728, 96), (9728, 2816, 216)])
@pytest.mark.parametrize("mv", [False, True])
@pytest.mark.parametrize("qtype", [12, 13, 14, 8])
def test_few_tokens_past_the_last_tile(M, monkeypatch, qtype, mv, rows, cols, tokens):  # noqa: F811
    """Sizes where the tokens past the last whole tile run as a product of their own."""
    w = M.synth_blocks(qtype, rows, rows, cols)
    x = M.synth_normal(rows, tokens * cols)
    res = M.synth_normal(tokens, tokens * rows) if mv else None
    ref = product(M, monkeypatch, {"MYNAH_GEMM_MFMA": "0"}, mv, qtype, w, rows, cols, x, tokens,
                  res)
    got = product(M, monkeypatch, {}, mv, qtype, w, rows, cols, x, tokens, res)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
