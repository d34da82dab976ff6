"""The MFMA GEMM's tiles, wave groups and splits (csrc/gemm_mfma.hip, planned
by csrc/matmat.c) where they can go wrong, bit for bit against the VALU
kernels of csrc/gemm_exact.hip (themselves held to the oracle by
tests/test_gemv_gpu.py and tests/test_prefill_gpu.py): rows and tokens around
the 16-row wave, the 64 x 64 tile and the four 16-token blocks, one to nine
super-blocks over one, two and four waves per row group, with and without
splits through memory; and blocks of any bit pattern, with non-finite
activations.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import mynah_amd
    mynah_amd.check(mynah_amd.lib.mynah_hip_init(0), "init")
    return mynah_amd


def product(M, monkeypatch, env, mv, qtype, w, rows, cols, x, tokens, res):
    for k in ("MYNAH_GEMM_MFMA", "MYNAH_GEMM_SPLIT", "MYNAH_GEMM_KW", "MYNAH_GEMM_FEW"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    wd, xd, yd = M.DeviceBuffer.from_array(w), M.DeviceBuffer.from_array(x), \
        M.DeviceBuffer(4 * rows * tokens)
    rd = M.DeviceBuffer.from_array(res) if res is not None else None
    try:
        if mv:
            M.check(M.lib.mynah_hip_matmat_mv_dev(qtype, wd.ptr, rows, cols, xd.ptr, yd.ptr,
                                                  tokens, rd.ptr if rd else None, None), "mv")
        else:
            M.check(M.lib.mynah_hip_matmat_dev(qtype, wd.ptr, rows, cols, xd.ptr, yd.ptr, tokens,
                                               None), "matmat")
        M.sync()
        return yd.download(np.float32, rows * tokens)
    finally:
        for b in (wd, xd, yd, rd):
            if b is not None:
                b.free()


def same(a, b):
    """Equal bits; NaNs by place (their payloads are not part of the result)."""
    return np.array_equal(np.isnan(a), np.isnan(b)) and \
        np.array_equal(a.view(np.uint32)[~np.isnan(a)], b.view(np.uint32)[~np.isnan(b)])


@pytest.mark.parametrize("rows,units,tokens", [
    (1, 1, 2), (15, 2, 15), (16, 3, 16), (17, 4, 17), (63, 5, 63), (64, 1, 64), (65, 9, 65),
    (130, 6, 81), (66, 7, 129)])
@pytest.mark.parametrize("mv", [False, True])
@pytest.mark.parametrize("qtype", [12, 13, 14, 8])
def test_tiles_and_wave_groups(M, monkeypatch, qtype, mv, rows, units, tokens):
    cols = 256 * units
    w = M.synth_blocks(qtype, rows, rows, cols)
    x = M.synth_normal(units, tokens * cols)
    res = M.synth_normal(tokens, tokens * rows) if mv else None
    ref = product(M, monkeypatch, {"MYNAH_GEMM_MFMA": "0"}, mv, qtype, w, rows, cols, x, tokens,
                  res)
    # Few tiles: the plan splits over super-blocks unless told not to. The full
    # tile also where at most 32 tokens would take kernels of their own
    # (MYNAH_GEMM_FEW=0).
    for env in ({}, {"MYNAH_GEMM_SPLIT": "0"}, {"MYNAH_GEMM_FEW": "0"},
                *({"MYNAH_GEMM_KW": k, "MYNAH_GEMM_SPLIT": s, "MYNAH_GEMM_FEW": "0"}
                  for k in "124" for s in "03")):
        got = product(M, monkeypatch, env, mv, qtype, w, rows, cols, x, tokens, res)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), env


@pytest.mark.parametrize("mv", [False, True])
@pytest.mark.parametrize("qtype", [12, 13, 14, 8])
def test_any_block_and_non_finite_activations(M, monkeypatch, qtype, mv):
    rows, cols, tokens = 70, 768, 66
    rng = np.random.default_rng(qtype)
    w = rng.integers(0, 256, rows * M.row_bytes(qtype, cols), dtype=np.uint8)
    x = rng.standard_normal((tokens, cols)).astype(np.float32)
    x[3, 5], x[9, 700], x[20, 255], x[21] = np.inf, -np.inf, np.nan, 0.0
    x[30] *= np.float32(1e-38)
    x[31] *= np.float32(3e37)
    x = x.reshape(-1)
    ref = product(M, monkeypatch, {"MYNAH_GEMM_MFMA": "0"}, mv, qtype, w, rows, cols, x, tokens,
                  None)
    for k in "124":
        env = {"MYNAH_GEMM_KW": k, "MYNAH_GEMM_FEW": "0"}
        assert same(product(M, monkeypatch, env, mv, qtype, w, rows, cols, x, tokens, None), ref)
