"""The one-launch exact attention of short contexts against the oracle.

Up to 256 positions one launch computes a query head's scores, softmax and
weighted sum (two passes of 128 positions, 16 per wave and pass). Bit-identical to the oracle's attention, the
logits and the key row it leaves in the cache, at the edges of the waves, the
passes, the unrolled chain (32 positions, then groups of four, then one to
three) and the 256-position line, for head groups 2 to 8; with the double sums
in index order throughout; and in steps replayed from a graph across the line.
"""
from __future__ import annotations

import numpy as np
import pytest

import configs as CF
import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import mynah_amd
    mynah_amd.check(mynah_amd.lib.mynah_hip_init(0), "init")
    mynah_amd.check(mynah_amd.lib.mynah_hip_set_gemv_order(0), "order")
    O.orc.orc_threads_init(0)
    return mynah_amd


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def make(M, group, n_pre, n_ctx):
    shape = CF.Qwen3Shape(1, 256, 256, 2 * group, 2, 128, 512)
    model = M.SynthQwen3(shape, 0)
    dec, orc = M.Qwen3Decoder(model, n_ctx), O.OracleQwen3(O.SynthModel(shape, 0), n_ctx)
    if n_pre:
        k, v = O.kv_prefill(O.substream, shape, 0, n_pre)
        dec.set_kv(k, v, n_pre)
        orc.prefill_kv(k, v, n_pre)
    return dec, orc


@pytest.mark.parametrize("index_sums", [0, 1])
@pytest.mark.parametrize("group", [2, 3, 4, 8])
@pytest.mark.parametrize("n_pre", [0, 1, 2, 3, 15, 30, 31, 32, 62, 127, 128, 144, 200, 253,
                                   255])
def test_steps_against_oracle(M, index_sums, group, n_pre):
    print(f"[case] group={group} n_pre={n_pre} index sums {index_sums}", flush=True)
    dec, orc = make(M, group, n_pre, 300)
    M.check(M.lib.mynah_hip_set_index_order_sums(index_sums), "index sums")
    try:
        for tok in (5, 77, 3):
            lg, want = dec.forward(tok), orc.forward(tok)
            assert np.array_equal(bits(dec.read_attn()), bits(orc.last_attn()))
            assert np.array_equal(bits(lg), bits(want))
    finally:
        M.check(M.lib.mynah_hip_set_index_order_sums(0), "index sums")
        dec.close()


@pytest.mark.parametrize("n_pre", [230, 250])
def test_replayed_steps_across_the_line(M, n_pre):
    inputs = np.arange(3, 23, dtype=np.int32)
    dec, orc = make(M, 2, n_pre, 300)
    _, lg = dec.forced(inputs)
    for tok in inputs:
        want = orc.forward(int(tok))
    assert np.array_equal(bits(lg), bits(want))
    dec.close()


def test_reset_and_shorter_context(M):
    """After a reset the launch's early loads cover positions past the new one."""
    dec, orc = make(M, 2, 200, 256)
    dec.forced(np.arange(1, 18, dtype=np.int32))
    dec.reset()
    orc = make(M, 2, 0, 256)[1]
    inputs = np.arange(40, 59, dtype=np.int32)
    _, lg = dec.forced(inputs)
    for tok in inputs:
        want = orc.forward(int(tok))
    assert np.array_equal(bits(lg), bits(want))
    dec.close()
